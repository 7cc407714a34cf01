"""GPU parity: k-means kernels and top-k selection (through the C ABI) against the CPU oracle.

Assignments must equal the oracle's fp64 arg-max except on near-ties: tokens whose best and second-best
scores differ by less than 1e-5 relative, where the fp32 MFMA accumulation may pick the other candidate.
Cluster sums are exact on both sides, so centroids computed from the same assignment must agree bit for
bit (one bf16 ulp is tolerated on at most 0.1 % of the components: the squared norm is reduced in a
different fp64 order before it is rounded to fp32).
"""
import math

import pytest
import torch

from oracle import inputs
from oracle import kmeans as KM

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NEAR_TIE = 1e-5


def _bf16_ulp_diff(a, b):
    ia = a.view(torch.int16).to(torch.int32)
    ib = b.view(torch.int16).to(torch.int32)
    return (ia - ib).abs()


@pytest.mark.parametrize("normalize", [True, False])
@pytest.mark.parametrize("G,N,C", [(2, 3000, 64), (1, 4096, 160), (1, 9000, 2048), (1, 20000, 8192)])
def test_train_step_teacher_forced(G, N, C, normalize):
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _triton_k_means_train

    print(f"case kmeans train G={G} N={N} C={C} normalize={normalize}", flush=True)
    key, _ = inputs.kmeans_inputs(G, N, 128, n_modes=24, seed=50 + C)
    cent0 = key[:, KM.init_centroid_indices(N, C)].clone()
    cent0[:, 7] = cent0[:, 6]                         # duplicate centroid: ties go to the lower index, 7 stays empty
    ref_idx, gap = KM.assign(key, cent0)
    cent_d = cent0.clone().to(DEV)
    _, idx_d, max_cnt = _triton_k_means_train(key.to(DEV), cent_d, normalize_centroids=normalize, return_indices=True)
    torch.cuda.synchronize()
    idx = idx_d.cpu()
    differ = idx != ref_idx
    assert bool((gap[differ] < NEAR_TIE).all()), f"{int(differ.sum())} assignments differ outside near-ties"
    assert int(differ.sum()) <= max(2, N // 2000)
    # centroids from the kernel's own assignment: exact sums -> same bits
    S, cnt = KM.cluster_sums(key, idx, C)
    assert max_cnt == int(cnt.max())
    exp = KM.update(cent0, S, cnt, normalize)
    got = cent_d.cpu()
    ulp = _bf16_ulp_diff(got, exp)
    assert int(ulp.max()) <= 1 and float((ulp > 0).float().mean()) <= 1e-3
    empty = cnt == 0
    assert bool(empty[:, 7].all()) and torch.equal(got[empty], cent0[empty])   # empty clusters keep the old centroid


def test_reverse_index_and_index_add_exact():
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import triton_index_add, triton_reverse_index

    G, N, C = 3, 5000, 96
    g = torch.Generator().manual_seed(3)
    idx = torch.randint(0, C, (G, N), generator=g, dtype=torch.int32)
    idx[idx == 11] = 12                                   # one empty cluster
    value = torch.randn(G, N, 128, generator=g).bfloat16()
    max_size = int(torch.stack([torch.bincount(idx[i].long(), minlength=C) for i in range(G)]).max())
    clusters, size = triton_reverse_index(idx.to(DEV), C, max_size)
    vsum = triton_index_add(value.to(DEV), idx.to(DEV), C)
    torch.cuda.synchronize()
    rc, rs = KM.reverse_index(idx, C, max_size)
    assert torch.equal(size.cpu(), rs) and torch.equal(clusters.cpu(), rc)
    assert torch.equal(vsum.cpu(), KM.index_add(value, idx, C))


def test_index_add_many_tiles_and_one_huge_cluster():
    """The grouping behind the sums works tile by tile: more tiles than one pass of the sum kernel walks (256), a ragged
    last tile, a cluster far larger than the id list the kernel stages at a time (the tiles sum its rows themselves), one
    with just under 2048 tokens per pass, an empty cluster.  Sums are exact."""
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import triton_index_add

    G, N, C = 1, 600_001, 32
    g = torch.Generator().manual_seed(17)
    idx = torch.randint(0, C, (G, N), generator=g, dtype=torch.int32)
    u = torch.rand(G, N, generator=g)
    idx[u < 0.5] = 3                                      # about 300 000 tokens in one cluster
    idx[(u >= 0.5) & (u < 0.5156)] = 9                    # about 64 per tile of 2048 tokens: either side of the size from which a tile sums a range itself
    idx[idx == 5] = 6
    value = torch.randn(G, N, 128, generator=g).bfloat16()
    vsum = triton_index_add(value.to(DEV), idx.to(DEV), C)
    torch.cuda.synchronize()
    assert torch.equal(vsum.cpu(), KM.index_add(value, idx, C))


@pytest.mark.parametrize("C", [8192, 5000, 1025])
def test_index_add_many_clusters(C):
    """Cluster counts up to the supported maximum (8192: the grouping kernel's counters, ids and long-range sums then
    take 72 KB of LDS, above the default limit; its prefix over the clusters runs in eight rounds) and counts that are
    not multiples of anything: sums exact, reverse index exact."""
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import triton_index_add, triton_reverse_index

    G, N = 2, 30_000
    g = torch.Generator().manual_seed(C)
    idx = torch.randint(0, C, (G, N), generator=g, dtype=torch.int32)
    idx[0, :3000] = C - 1                                  # one long range at the last cluster
    value = torch.randn(G, N, 128, generator=g).bfloat16()
    vsum = triton_index_add(value.to(DEV), idx.to(DEV), C)
    msize = int(torch.stack([torch.bincount(idx[i].long(), minlength=C) for i in range(G)]).max())
    clusters, size = triton_reverse_index(idx.to(DEV), C, msize)
    torch.cuda.synchronize()
    assert torch.equal(vsum.cpu(), KM.index_add(value, idx, C))
    rc, rs = KM.reverse_index(idx, C, msize)
    assert torch.equal(size.cpu(), rs) and torch.equal(clusters.cpu(), rc)


@pytest.mark.parametrize("segments", [1, 2])
def test_segment_k_means_end_to_end(segments):
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import segment_k_means

    G, N, C = 2, 4096, 64
    key, value = inputs.kmeans_inputs(G, N, 128, n_modes=20, seed=61)
    cent, vsum, clusters, size = segment_k_means(key.to(DEV), value.to(DEV), C, num_iters=4, num_segments=segments)
    torch.cuda.synchronize()
    rcent, rvsum, rclusters, rsize = KM.segment_k_means(key, value, C, num_iters=4, num_segments=segments)
    size, clusters = size.cpu(), clusters.cpu()
    assert int(size.sum()) == G * N
    for g in range(G):
        toks = torch.cat([clusters[g, c, : int(size[g, c])] for c in range(C)])
        assert torch.equal(torch.sort(toks).values, torch.arange(N, dtype=torch.int32))
    # free-running iterations: identical unless a near-tie flipped somewhere along the way
    own = torch.empty(G, N, dtype=torch.int64)
    ref = torch.empty(G, N, dtype=torch.int64)
    for g in range(G):
        for c in range(C):
            own[g, clusters[g, c, : int(size[g, c])].long()] = c
            ref[g, rclusters[g, c, : int(rsize[g, c])].long()] = c
    assert float((own == ref).float().mean()) >= 0.999
    ulp = _bf16_ulp_diff(cent.cpu(), rcent)
    assert float((ulp <= 1).float().mean()) >= 0.99
    assert torch.allclose(vsum.cpu().float(), rvsum.float(), atol=0.5, rtol=0.05) or float((own == ref).float().mean()) < 1.0


def test_topk_select_matches_oracle():
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import topk_select

    B, Hq, groups, N, C, k = 2, 8, 4, 2048, 64, 700
    Hkv = Hq // groups
    key, value = inputs.kmeans_inputs(B * Hkv, N, 128, n_modes=20, seed=71)
    cent, _, clusters, size = KM.segment_k_means(key, value, C, num_iters=3)
    q = torch.randn(B, Hq, 128, generator=torch.Generator().manual_seed(2)).bfloat16()
    sel = topk_select(q.to(DEV), cent.to(DEV), clusters.to(DEV), size.to(DEV), k, groups)
    torch.cuda.synchronize()
    assert torch.equal(sel.cpu(), KM.topk_select(q, cent, clusters, size, k, groups))
    # k larger than the number of tokens: the tail is -1
    sel2 = topk_select(q.to(DEV), cent.to(DEV), clusters.to(DEV), size.to(DEV), N + 50, groups).cpu()
    assert bool((sel2[:, N:] == -1).all()) and bool((sel2[:, :N] >= 0).all())
    for g in range(B * Hkv):
        assert torch.equal(torch.sort(sel2[g, :N]).values, torch.arange(N, dtype=torch.int32))


def test_topk_select_shared_score_phase_repeated():
    """With 1024 clusters several workgroups share a head's score phase and the last to arrive finishes the selection,
    handing the scores over through memory.  Two queries alternate over 1000 calls; every call must reproduce its query's
    oracle result exactly (a score that arrives late, or a counter that is not set back, would show)."""
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _workspace, topk_select

    B, Hkv, groups, N, C, k = 2, 4, 7, 8192, 1024, 1000
    G = B * Hkv
    g = torch.Generator().manual_seed(81)
    idx = torch.randint(0, C, (G, N), generator=g, dtype=torch.int32)
    msize = int(torch.stack([torch.bincount(idx[i].long(), minlength=C) for i in range(G)]).max())
    clusters, size = KM.reverse_index(idx, C, msize)
    cent = torch.randn(G, C, 128, generator=g).bfloat16()
    qs = [torch.randn(B, Hkv * groups, 128, generator=g).bfloat16() for _ in range(2)]
    want = [KM.topk_select(q, cent, clusters, size, k, groups) for q in qs]
    dq = [q.to(DEV) for q in qs]
    dc, dcl, dsz = cent.to(DEV), clusters.to(DEV), size.to(DEV)
    ws = _workspace(G, 1, C, DEV)   # one workspace for all calls: a stale score would be the other query's
    outs = [topk_select(dq[i % 2], dc, dcl, dsz, k, groups, workspace=ws) for i in range(1000)]
    torch.cuda.synchronize()
    for i, o in enumerate(outs):
        assert torch.equal(o.cpu(), want[i % 2]), i


def _shared_phase_case(seed):
    B, Hkv, groups, N, C, k = 1, 4, 7, 8192, 1024, 1000
    g = torch.Generator().manual_seed(seed)
    idx = torch.randint(0, C, (B * Hkv, N), generator=g, dtype=torch.int32)
    msize = int(torch.stack([torch.bincount(idx[i].long(), minlength=C) for i in range(B * Hkv)]).max())
    clusters, size = KM.reverse_index(idx, C, msize)
    cent = torch.randn(B * Hkv, C, 128, generator=g).bfloat16()
    q = torch.randn(B, Hkv * groups, 128, generator=g).bfloat16()
    return q, cent, clusters, size, k, groups


@pytest.mark.parametrize("fill", ["ones", "random", "finished", "other_shape"])
def test_topk_select_tagged_words_need_no_initialisation(fill):
    """The tagged score words of the shared score phase live in the caller's workspace and are never cleared by the host.
    Whatever the memory holds -- all bits set, random words, the words a finished call leaves, or those of a call
    with another number of heads -- the first call over it must select what the oracle selects."""
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _workspace, topk_select

    q, cent, clusters, size, k, groups = _shared_phase_case(83)
    G, C = cent.shape[0], cent.shape[1]
    want = KM.topk_select(q, cent, clusters, size, k, groups)
    ws = _workspace(G, 1, C, DEV)
    words = ws[: ws.numel() // 4 * 4].view(torch.int32)
    if fill == "ones":
        ws.fill_(0xFF)
    elif fill == "random":
        words.copy_(torch.randint(-2**31, 2**31 - 1, (words.numel(),), generator=torch.Generator().manual_seed(5),
                                  dtype=torch.int64).to(torch.int32).to(DEV))
    elif fill == "finished":
        topk_select(q.to(DEV), cent.to(DEV), clusters.to(DEV), size.to(DEV), k, groups, workspace=ws)
    else:   # a call over 2 of the 4 heads first, then all 4 over the same memory
        topk_select(q[:, : 2 * groups].to(DEV), cent[:2].to(DEV), clusters[:2].to(DEV), size[:2].to(DEV), k, groups,
                    workspace=ws)
    for _ in range(3):
        got = topk_select(q.to(DEV), cent.to(DEV), clusters.to(DEV), size.to(DEV), k, groups, workspace=ws)
        torch.cuda.synchronize()
        assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("C", [64, 1000, 1024])
@pytest.mark.parametrize("pattern", ["equal", "outlier", "binades", "infinite", "zeros", "falling"])
def test_topk_select_score_patterns(pattern, C):
    """Scores that strain the histogram between the extremes: all equal, one far above the rest, a range of 2^60, infinities
    (no finite range), +0 beside -0, and one value per bin.  The scores are exact, so the ids are the oracle's, bit for bit."""
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import topk_select

    print(f"case topk pattern {pattern} C={C}", flush=True)
    g = torch.Generator().manual_seed(7 * C + len(pattern))
    B, groups, Hkv = 1, 3, 2
    G = B * Hkv
    x = torch.randn(G, C, generator=g)
    if pattern == "equal":
        x.fill_(1.5)
    elif pattern == "outlier":
        x[:, C // 3] = 1e30
    elif pattern == "binades":
        x = torch.sign(x) * torch.exp2(torch.randint(-30, 31, (G, C), generator=g).float())
    elif pattern == "infinite":
        x[:, ::7] = float("inf")
        x[:, 3::11] = float("-inf")
    elif pattern == "zeros":
        x = torch.where(x > 0.5, x, torch.where(x > 0, 0.0, -0.0))
    else:
        x = (C - torch.arange(C).float()).expand(G, C)
    cent = torch.zeros(G, C, 128)
    cent[..., 0] = x
    q = torch.zeros(B, Hkv * groups, 128)
    q[..., 0] = 1.0
    cent, q = cent.bfloat16(), q.bfloat16()
    size = torch.randint(0, 40, (G, C), generator=g, dtype=torch.int32)   # empty clusters among them
    clusters = torch.randint(0, 100000, (G, C, 40), generator=g, dtype=torch.int32)
    total = int(size.sum(dim=1).max())
    for k in (1, 511, total // 2, total + 9):
        got = topk_select(q.to(DEV), cent.to(DEV), clusters.to(DEV), size.to(DEV), k, groups)
        assert torch.equal(got.cpu(), KM.topk_select(q, cent, clusters, size, k, groups)), k


@pytest.mark.parametrize("C", [64, 1000, 1024, 1100])
@pytest.mark.parametrize("groups", [1, 3, 16])
def test_topk_select_scores_that_are_not_numbers_come_last(C, groups):
    """A NaN score never wins a maximum: a cluster whose centroid holds one ranks with -inf, behind every number (ties by index), a
    query head that holds one is out of the maximum.  By every route: one workgroup, a shared score phase, two kernels."""
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import topk_select

    print(f"case topk NaN C={C} groups={groups}", flush=True)
    g = torch.Generator().manual_seed(C + groups)
    Hkv = 2
    cent, q = torch.zeros(Hkv, C, 128), torch.zeros(1, Hkv * groups, 128)
    cent[..., 0] = torch.randn(Hkv, C, generator=g)
    q[..., 0] = 1.0
    size = torch.randint(0, 9, (Hkv, C), generator=g, dtype=torch.int32)
    clusters = torch.randint(0, 100000, (Hkv, C, 9), generator=g, dtype=torch.int32)
    want_cent = cent.clone()
    cent[:, ::5, 0], want_cent[:, ::5, 0] = float("nan"), float("-inf")
    cent[:, 3, 0], want_cent[:, 3, 0] = float("-inf"), float("-inf")
    want_q = q.clone()
    if groups > 1:
        q[0, 1] = float("nan")
        want_q[0, 1] = q[0, 0]
    cent, q, want_cent, want_q = (t.bfloat16() for t in (cent, q, want_cent, want_q))
    cent.view(torch.int16)[:, ::10, 0] ^= -32768   # NaNs of either sign
    total = int(size.sum(dim=1).max())
    for k in (7, total // 3, total + 5):
        got = topk_select(q.to(DEV), cent.to(DEV), clusters.to(DEV), size.to(DEV), k, groups)
        assert torch.equal(got.cpu(), KM.topk_select(want_q, want_cent, clusters, size, k, groups)), k


@pytest.mark.parametrize("B", [1, 16, 25, 80])
def test_topk_select_replayed_from_a_graph(B):
    """4 B heads share the score phase two, four, eight or sixteen waves a workgroup.  One captured call, replayed over another
    query each time, with the workspace as the replay before left it and overwritten in between: the oracle's ids every time."""
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _workspace, topk_select

    print(f"case topk graph B={B}", flush=True)
    Hkv, groups, C, M, k = 4, 2, 1024, 8, 37
    G = B * Hkv
    g = torch.Generator().manual_seed(B)
    size = torch.randint(0, M + 1, (G, C), generator=g, dtype=torch.int32)
    clusters = torch.randint(0, 100000, (G, C, M), generator=g, dtype=torch.int32)
    cent = torch.randn(G, C, 128, generator=g).bfloat16()
    qs = [torch.randn(B, Hkv * groups, 128, generator=g).bfloat16() for _ in range(4)]
    dq, dc, dcl, dsz = qs[0].to(DEV), cent.to(DEV), clusters.to(DEV), size.to(DEV)
    ws = _workspace(G, 1, C, DEV)
    out = torch.empty(G, k, dtype=torch.int32, device=DEV)
    topk_select(dq, dc, dcl, dsz, k, groups, out=out, workspace=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        topk_select(dq, dc, dcl, dsz, k, groups, out=out, workspace=ws)
    for i, q in enumerate(qs):
        dq.copy_(q)
        if i == 2:
            ws.view(torch.int32).random_()
        out.fill_(-7)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), KM.topk_select(q, cent, clusters, size, k, groups)), i


def test_topk_select_two_workspaces_on_two_streams():
    """Calls that use different workspaces share nothing: two selections with different queries run on two streams at
    the same time, 200 times, and each must equal its own oracle result."""
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _workspace, topk_select

    cases = [_shared_phase_case(s) for s in (85, 86)]
    want = [KM.topk_select(*c) for c in cases]
    dev = [[x.to(DEV) if torch.is_tensor(x) else x for x in c] for c in cases]
    G, C = cases[0][1].shape[0], cases[0][1].shape[1]
    wss = [_workspace(G, 1, C, DEV) for _ in cases]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    outs = [[], []]
    for _ in range(200):
        for i in (0, 1):
            with torch.cuda.stream(streams[i]):
                outs[i].append(topk_select(*dev[i], workspace=wss[i]))
    torch.cuda.synchronize()
    for i in (0, 1):
        for o in outs[i]:
            assert torch.equal(o.cpu(), want[i])


def test_full_size_properties():
    """Benchmark shape (4 heads x 131072 tokens x 128, 1024 centroids): size-independent invariants plus an
    oracle check on a token sample."""
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _triton_k_means_train, triton_reverse_index

    G, N, C = 4, 131072, 1024
    key, _ = inputs.kmeans_inputs(G, N, 128, seed=4)
    cent0 = key[:, KM.init_centroid_indices(N, C)].clone()
    kd, cd = key.to(DEV), cent0.clone().to(DEV)
    _, idx_d, max_cnt = _triton_k_means_train(kd, cd, normalize_centroids=True, return_indices=True)
    clusters, size = triton_reverse_index(idx_d, C, max_cnt)
    torch.cuda.synchronize()
    idx, size = idx_d.cpu(), size.cpu()
    assert int(size.sum()) == G * N and int(size.max()) == max_cnt
    for g in range(G):
        assert torch.equal(size[g].long(), torch.bincount(idx[g].long(), minlength=C))
    flat = clusters.cpu()
    for g in range(G):
        mask = torch.arange(flat.shape[2])[None, :] < size[g][:, None]
        assert torch.equal(torch.sort(flat[g][mask]).values, torch.arange(N, dtype=torch.int32))
    sample = slice(5000, 5000 + 4096)
    ref_idx, gap = KM.assign(key[:, sample], cent0)
    differ = idx[:, sample] != ref_idx
    assert bool((gap[differ] < NEAR_TIE).all())
    nrm = cd.cpu()[size > 0].float().norm(dim=-1)
    assert float((nrm - 1).abs().max()) < 1e-2


def test_kmeans_configurations_drawn_at_random():
    """A seeded sweep over the training step and the index helpers: 1 to 5 groups, token counts that are not multiples of the
    256-token tile (down to fewer tokens than centroids), centroid counts from 32 to 1056 (multiples of 32, with and
    without a half block at the end), normalised or not -- each against the oracle under the rules at the top."""
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _triton_k_means_train, triton_index_add, triton_reverse_index

    rng = torch.Generator().manual_seed(99)

    def pick(options):
        return options[int(torch.randint(0, len(options), (1,), generator=rng))]

    for case in range(12):
        G = pick([1, 2, 3, 5])
        C = 32 * pick([1, 2, 3, 5, 8, 17, 33])
        N = int(torch.randint(max(40, C // 2), 6000, (1,), generator=rng))
        normalize = bool(case % 2)
        print(f"case kmeans #{case}: G={G} N={N} C={C} normalize={normalize}", flush=True)
        key, value = inputs.kmeans_inputs(G, N, 128, n_modes=min(C, 40), seed=600 + case)
        cent0 = key[:, torch.randint(0, N, (C,), generator=rng)].clone()   # repeated picks give duplicate centroids
        ref_idx, gap = KM.assign(key, cent0)
        cent_d = cent0.clone().to(DEV)
        _, idx_d, max_cnt = _triton_k_means_train(key.to(DEV), cent_d, normalize_centroids=normalize, return_indices=True)
        torch.cuda.synchronize()
        idx = idx_d.cpu()
        differ = idx != ref_idx
        assert bool((gap[differ] < NEAR_TIE).all()), (case, int(differ.sum()))
        S, cnt = KM.cluster_sums(key, idx, C)
        assert max_cnt == int(cnt.max())
        ulp = _bf16_ulp_diff(cent_d.cpu(), KM.update(cent0, S, cnt, normalize))
        assert int(ulp.max()) <= 1 and float((ulp > 0).float().mean()) <= 1e-3, case
        clusters, size = triton_reverse_index(idx_d, C, max_cnt)
        vsum = triton_index_add(value.to(DEV), idx_d, C)
        torch.cuda.synchronize()
        rc, rs = KM.reverse_index(idx, C, max_cnt)
        assert torch.equal(size.cpu(), rs) and torch.equal(clusters.cpu(), rc), case
        assert torch.equal(vsum.cpu(), KM.index_add(value, idx, C)), case


@pytest.mark.parametrize("G,N,C,modes", [(2, 5000, 64, 20), (1, 40000, 1024, 300), (3, 777, 32, 5)])
def test_carried_sums_give_the_bits_of_the_full_resum(G, N, C, modes):
    """`sq_kmeans_train_stateful`: a run of Lloyd steps whose cluster sums are carried in the workspace (one step that
    keeps them, then steps that only apply the tokens that changed cluster) against the same run with every step
    re-summing every row.  The sums are exact, so centroids, assignment and sizes must be equal bit for bit after every
    step -- normalised and un-normalised steps, empty clusters, N not a multiple of the 256-token tile, and a step in
    which nothing moves."""
    from longcontext_sqattn_paddle_amd import _native as NV
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _triton_k_means_train, _workspace

    print(f"case k-means carried sums G={G} N={N} C={C}", flush=True)
    key, _ = inputs.kmeans_inputs(G, N, 128, n_modes=modes, seed=70 + C)
    data = key.to(DEV)
    sel = KM.init_centroid_indices(N, C).to(DEV)
    ca, cb = data.index_select(1, sel).contiguous(), data.index_select(1, sel).contiguous()
    ia = torch.empty(G, N, dtype=torch.int32, device=DEV)
    ib = torch.full((G, N), -7, dtype=torch.int32, device=DEV)
    wa, wb = _workspace(G, N, C, DEV), _workspace(G, N, C, DEV)
    wb.fill_(0x5A)      # whatever the workspace held before must not matter
    moved = []
    for step in range(9):
        norm = step != 5                                   # one un-normalised step in the middle of the run
        state = NV.KMEANS_STATELESS if step == 0 else (NV.KMEANS_KEEP_SUMS if step == 1 else NV.KMEANS_APPLY_CHANGES)
        prev = ib.clone()
        _, _, max_a = _triton_k_means_train(data, ca, max_idx=ia, normalize_centroids=norm, return_indices=True, workspace=wa)
        _, _, max_b = _triton_k_means_train(data, cb, max_idx=ib, normalize_centroids=norm, return_indices=True, workspace=wb, state=state)
        torch.cuda.synchronize()
        moved.append(int((prev != ib).sum()))
        assert torch.equal(ia, ib), step
        assert torch.equal(ca.view(torch.int16), cb.view(torch.int16)), step
        assert max_a == max_b, step
    print(f"  tokens that changed cluster per step: {moved}", flush=True)
    # a step in which nothing moves (the same centroids again cannot be had, but the same assignment can: feed the
    # centroids of the stateless run, which are equal, and repeat until the assignment is stable or 20 steps have passed)
    for _ in range(20):
        prev = ib.clone()
        _triton_k_means_train(data, ca, max_idx=ia, normalize_centroids=True, workspace=wa)
        _triton_k_means_train(data, cb, max_idx=ib, normalize_centroids=True, workspace=wb, state=NV.KMEANS_APPLY_CHANGES)
        torch.cuda.synchronize()
        assert torch.equal(ia, ib) and torch.equal(ca.view(torch.int16), cb.view(torch.int16))
        if torch.equal(prev, ib):
            break
    # the sizes the carried state reports are the histogram of the assignment
    cnt = torch.empty(G, C, dtype=torch.int32, device=DEV)
    b = [NV.dl(t) for t in (data, cb, ib, cnt, wb)]
    NV.check(NV.lib().sq_kmeans_train_stateful(*[NV.ptr(x) for x in b], 1, NV.KMEANS_APPLY_CHANGES, NV.current_stream(data.device)))
    torch.cuda.synchronize()
    for g in range(G):
        assert torch.equal(cnt[g].cpu().long(), torch.bincount(ib[g].cpu().long(), minlength=C))


def test_segment_k_means_with_carried_sums_equals_stateless_steps():
    """`segment_k_means` carries the sums from its fourth step on; written out with stateless steps only it must return
    the same centroids, value sums, clusters and sizes (one segment, where the last step continues the carried run, and
    two, where it starts over on the unsegmented data)."""
    from longcontext_sqattn_paddle_amd.cache_hub import kmeans as HK

    key, value = inputs.kmeans_inputs(2, 6000, 128, n_modes=40, seed=81)
    key, value = key.to(DEV), value.to(DEV)
    for segments in (1, 2):
        got = HK.segment_k_means(key, value, 64, num_iters=8, num_segments=segments)
        saved, HK.FULL_RESUM_STEPS = HK.FULL_RESUM_STEPS, 1 << 30       # every step stateless
        try:
            want = HK.segment_k_means(key, value, 64, num_iters=8, num_segments=segments)
        finally:
            HK.FULL_RESUM_STEPS = saved
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert a.shape == b.shape and torch.equal(a.view(torch.int16) if a.dtype == torch.bfloat16 else a, b.view(torch.int16) if b.dtype == torch.bfloat16 else b), segments


def _parts(G, N, C):
    """Shares of the centroids per workgroup (launch_assign): 64-token workgroups with four while 256 of them do, 128-token ones
    with two while 256 do, else 256-token ones; one up to 128 tokens of up to three blocks of 64 centroids; from 32 groups on
    half as many workgroups, unless the chain of blocks is long."""
    blocks = -(-C // 64)
    if blocks == 1 or (blocks <= 3 and N <= 128):
        return 1
    if G * -(-N // 64) <= (256 if G < 32 or blocks >= 16 else 128):
        return 4
    return 2 if G * -(-N // 128) <= (256 if G < 32 or blocks >= 8 else 128) else 1


@pytest.mark.parametrize("G,N,C,parts", [(1, 1, 256, 4), (1, 63, 224, 4), (1, 65, 320, 4), (1, 129, 96, 4), (1, 200, 160, 4), (3, 257, 1024, 4), (1, 4097, 320, 4),
                                         (1, 16384, 96, 4), (1, 16385, 160, 2), (2, 16384, 1024, 2), (32, 256, 256, 4), (32, 257, 160, 2), (32, 512, 1024, 4),
                                         (32, 1000, 512, 2)])
def test_split_centroids_give_the_bits_of_the_unsplit_launch(G, N, C, parts):
    """The same groups alone and among so many copies that the launch is not split: assignments, centroids and sizes are equal
    to the bit, in the step that re-sums every row and in the two that carry the sums."""
    from longcontext_sqattn_paddle_amd import _native as NAT
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _triton_k_means_train, _workspace

    print(f"case kmeans split G={G} N={N} C={C} parts={parts}", flush=True)
    g = torch.Generator().manual_seed(90 + C)
    key = torch.randn(G, N, 128, generator=g).bfloat16()
    key[:, N // 2] = 0                                             # every score equal: index 0
    cent = torch.randn(G, C, 128, generator=g).bfloat16()
    cent[:, C - 1] = cent[:, C // 2] = cent[:, 1]                  # the same centroid in several shares: the lowest index wins
    copies = 1
    while _parts(copies * G, N, C) > 1:
        copies *= 2
    assert _parts(G, N, C) == parts > 1 and copies > 1
    small, large = [], []
    for reps, out in ((1, small), (copies, large)):
        kd, cd = key.repeat(reps, 1, 1).to(DEV), cent.repeat(reps, 1, 1).to(DEV)
        idx = torch.full((kd.shape[0], N), -1, dtype=torch.int32, device=DEV)
        ws = _workspace(kd.shape[0], N, C, DEV)
        for state in (NAT.KMEANS_STATELESS, NAT.KMEANS_KEEP_SUMS, NAT.KMEANS_APPLY_CHANGES, NAT.KMEANS_APPLY_CHANGES):
            _triton_k_means_train(kd, cd, max_idx=idx, workspace=ws, state=state)
            out += [idx[:G].cpu(), cd[:G].cpu().view(torch.int16)]
    assert int(small[0][:, N // 2].max()) == 0
    assert not bool(((small[0] == C - 1) | (small[0] == C // 2)).any())
    for a, b in zip(small, large):
        assert torch.equal(a, b)


@pytest.mark.parametrize("G,N,C,parts", [(2, 200, 320, 4), (1, 16400, 160, 2)])
def test_split_centroids_with_special_values(G, N, C, parts):
    """NaN keys (no score above -inf), extreme elements of keys, infinite and extreme ones of centroids (whole shares of centroids
    without a finite score among them): the assignments of the unsplit launch."""
    from longcontext_sqattn_paddle_amd import _native as NAT
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _triton_k_means_train, _workspace

    print(f"case kmeans split special values G={G} N={N} C={C} parts={parts}", flush=True)
    g = torch.Generator().manual_seed(17)
    key = torch.randn(G, N, 128, generator=g).bfloat16()
    cent = torch.randn(G, C, 128, generator=g).bfloat16()
    special = torch.tensor([1e37, -1e37, 1e30, -0.0, 1e-40]).bfloat16()
    key[:, :50, 3] = special[torch.randint(0, 5, (G, 50), generator=g)]
    key[:, 60:70] = math.nan
    cent[:, : C // 4, 9] = -math.inf                               # half of the tokens score -inf, the other half +inf
    cent[:, C // 2: C // 2 + 70, 11] = 3.3e38
    copies = 1
    while _parts(copies * G, N, C) > 1:
        copies *= 2
    assert _parts(G, N, C) == parts and copies > 1
    got = []
    for reps in (1, copies):
        kd, cd = key.repeat(reps, 1, 1).to(DEV), cent.repeat(reps, 1, 1).to(DEV)
        idx = torch.full((kd.shape[0], N), -1, dtype=torch.int32, device=DEV)
        _triton_k_means_train(kd, cd, max_idx=idx, workspace=_workspace(kd.shape[0], N, C, DEV), state=NAT.KMEANS_STATELESS)
        got.append(idx[:G].cpu())
    assert int(got[1].min()) >= 0 and int(got[1].max()) < C
    assert torch.equal(got[0], got[1])


def _bounded_data(G, N, C, kind, seed):
    """Rows around C / 2 centres, apart enough that the bounds leave most centroids out, and what they must not be misled by."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    mu = torch.randn(G, max(4, C // 2), 128, device=DEV, generator=g)
    which = torch.randint(0, mu.shape[1], (G, N), device=DEV, generator=g)
    sigma = {"overlap": 2.0, "half": 0.6}.get(kind, 0.3)
    x = torch.gather(mu, 1, which[..., None].expand(G, N, 128)) + sigma * torch.randn(G, N, 128, device=DEV, generator=g)
    if kind == "same":
        x = x[:, :1].expand(G, N, 128)
    if kind == "pairs":    # every row twice: ties wherever both copies are seeds
        x = x[:, torch.arange(N, device=DEV) // 2]
    if kind == "zero":
        x[:, ::5] = 0.0
    if kind == "nan":
        x[0, N // 3, 7] = math.nan
        x[-1, N // 2] = math.nan
    if kind == "inf":
        x[0, N // 3, 7] = math.inf
        x[-1, N // 2, 3] = -math.inf
    if kind in ("huge", "small", "tiny"):
        x = x * {"huge": 1e18, "small": 1e-7, "tiny": 1e-20}[kind]
    if kind in ("faint", "faint_means"):   # squares at and below the smallest 32-bit numbers
        x = x * 1e-23
    if kind == "signs":
        x = 2.5e-23 * x.sign()
    if kind == "offset":
        x = x + 40.0
    if kind == "one_sided":   # scores of both signs
        x[:, ::2] = -x[:, ::2]
    return x.bfloat16().contiguous()


BOUNDED_KINDS = ["apart", "half", "overlap", "same", "pairs", "zero", "nan", "inf", "huge", "small", "tiny", "faint", "faint_means", "signs",
                 "offset", "one_sided"]


# (257 tokens for 2048 centroids: a NaN token seeds eight neighbouring centroids, and what a token without a comparable score gets then
# already differs between the split and the unsplit assignment)
@pytest.mark.parametrize("G,N,C,kind", [(G, N, C, kind) for G, N, C in [(2, 700, 64), (1, 257, 2048), (3, 5000, 1056), (2, 12289, 512), (1, 40, 32), (3, 40000, 512),
                                                             (3, 12001, 1056), (1, 33000, 2048), (64, 1000, 96)]
                                        for kind in BOUNDED_KINDS if not (C > N and kind in ("nan", "inf"))])
def test_bounded_steps_have_the_bits_of_stateful_ones(G, N, C, kind):
    """`sq_kmeans_train_bounded` against `sq_kmeans_train_stateful`: assignment, centroids and sizes after every step, sizes at the
    edges of its tiles and lists.  One step starts from centroids that somebody else has changed in between."""
    from longcontext_sqattn_paddle_amd import _native as NV
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _triton_k_means_train, _workspace

    print(f"case bounded k-means G={G} N={N} C={C} {kind}", flush=True)
    data = _bounded_data(G, N, C, kind, 7 * N + C)
    seeds = (torch.arange(C, device=DEV) * N // C) % N
    ca = data[:, seeds].contiguous()
    cb = ca.clone()
    ia, ib = (torch.zeros(G, N, dtype=torch.int32, device=DEV) for _ in range(2))
    wa, wb = _workspace(G, N, C, DEV), _workspace(G, N, C, DEV, bounded=True)
    wb.view(torch.uint8).fill_(0xA5)
    for step in range(7):
        state = NV.KMEANS_STATELESS if step == 0 else (NV.KMEANS_KEEP_SUMS if step == 1 else NV.KMEANS_APPLY_CHANGES)
        if step == 4:
            for c in (ca, cb):
                c.copy_(c.roll(3, dims=1))
        norm = step < 6 and kind != "faint_means"
        ra = _triton_k_means_train(data, ca, max_idx=ia, normalize_centroids=norm, return_indices=True, workspace=wa, state=state)
        rb = _triton_k_means_train(data, cb, max_idx=ib, normalize_centroids=norm, return_indices=True, workspace=wb, state=state, bounded=True)
        assert torch.equal(ia, ib), (step, int((ia != ib).sum()))
        assert torch.equal(ca.view(torch.int16), cb.view(torch.int16)), step
        assert ra[2] == rb[2]


def _walks_everything(workspace, G):
    """The bounded form's own answer, out of the end of its workspace: nothing is left out any more."""
    return int(workspace[-((6 + G) * 4) // 256 * 256:].view(torch.int32)[4]) == 1


def _run_bounded(data, C, steps=8):
    from longcontext_sqattn_paddle_amd import _native as NV
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _triton_k_means_train, _workspace

    G, N, _ = data.shape
    cent = data[:, (torch.arange(C, device=DEV) * N // C) % N].contiguous()
    idx = torch.zeros(G, N, dtype=torch.int32, device=DEV)
    ws = _workspace(G, N, C, DEV, bounded=True)
    ws.fill_(0xA5)
    for step in range(steps):
        state = NV.KMEANS_STATELESS if step < 2 else (NV.KMEANS_KEEP_SUMS if step == 2 else NV.KMEANS_APPLY_CHANGES)
        _triton_k_means_train(data, cent, max_idx=idx, workspace=ws, state=state, bounded=True)
    torch.cuda.synchronize()
    return ws


# (64 groups of 4 tokens a cluster: short masks, but a workgroup's tokens are in 64 clusters)
@pytest.mark.parametrize("G,N,C,kind,all_walked", [(3, 12001, 1056, "overlap", True), (3, 12001, 1056, "apart", False), (1, 33000, 2048, "apart", False),
                                                   (3, 40000, 512, "apart", False), (2, 9001, 64, "apart", False), (64, 4096, 1024, "apart", True)])
def test_bounded_steps_leave_centroids_out_where_that_is_less_work(G, N, C, kind, all_walked):
    print(f"case bounded k-means, what is walked G={G} N={N} C={C} {kind}", flush=True)
    assert _walks_everything(_run_bounded(_bounded_data(G, N, C, kind, 7 * N + C), C), G) == all_walked


@pytest.mark.parametrize("G,N,C", [(1, 4096, 1024), (3, 5000, 1056), (2, 12289, 512)])
def test_bounded_steps_are_the_stateful_ones_where_these_split_the_centroids(G, N, C):
    """Up to about 32768 tokens: the workspace behind the stateful entry's stays as it was."""
    from longcontext_sqattn_paddle_amd import _native as NV

    print(f"case bounded k-means of few tokens G={G} N={N} C={C}", flush=True)
    ws = _run_bounded(_bounded_data(G, N, C, "apart", 3), C)
    assert bool((ws[NV.lib().sq_kmeans_workspace_bytes(G, N, C, 128):] == 0xA5).all())


def test_bounded_steps_refuse_more_centroids_than_their_lists_hold():
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import _triton_k_means_train

    data = torch.zeros(1, 100, 128, dtype=torch.bfloat16, device=DEV)
    cent = torch.zeros(1, 2080, 128, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError, match="more than 2048"):
        _triton_k_means_train(data, cent, bounded=True)


# (two segments of an odd number of tokens: the last step starts over, on all tokens and a workspace of its own)
@pytest.mark.parametrize("G,N,C,iters,segments", [(3, 40000, 1024, 8, 1), (2, 80001, 2048, 9, 2), (2, 80000, 2048, 10, 4), (1, 4096, 1024, 8, 1)])
@pytest.mark.parametrize("kind", ["apart", "overlap"])
def test_segment_k_means_is_the_same_with_and_without_bounds(monkeypatch, G, N, C, iters, segments, kind):
    from longcontext_sqattn_paddle_amd.cache_hub import kmeans as HK

    print(f"case segment_k_means with and without bounds G={G} N={N} C={C} iters={iters} segments={segments} {kind}", flush=True)
    key = _bounded_data(G, N, C, kind, N + C)
    value = torch.randn(key.shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(N)).bfloat16()
    step, steps = HK._step, []
    monkeypatch.setattr(HK, "_step", lambda *a: (steps.append(a[-1]), step(*a))[1])
    got = {}
    for bounded in (False, True):
        monkeypatch.setattr(HK, "_bounded", lambda *a: bounded)
        got[bounded] = HK.segment_k_means(key, value, C, iters, segments)
    assert steps == [False] * iters + [True] * (iters - (segments > 1)) + [False] * (segments > 1)
    for a, b in zip(got[False], got[True]):
        assert torch.equal(a, b)
