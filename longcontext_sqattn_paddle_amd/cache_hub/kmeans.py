"""KV k-means of the reference's cache_hub/kmeans.py on the gfx950 kernels (same function names).

`segment_k_means(key, value, num_centroids, num_iters=10, num_segments=1)` returns
`(centroids, value_sum, clusters, cluster_size)` exactly like the reference (:332-375).  Differences:
cluster sums are exact (fp64) instead of fp32 atomics in arbitrary order, and tokens inside a cluster are
listed in ascending order instead of arbitrary order.  `topk_select` has no reference counterpart.
"""
from __future__ import annotations

from typing import Optional

import torch

from .. import _native as N


def _require(t, what):
    if not t.is_cuda:
        raise RuntimeError(f"{what} must live on the MI355X (got {t.device}); there is no CPU path")


def _workspace(G: int, num_tokens: int, num_centroids: int, device, bounded: bool = False) -> torch.Tensor:
    size = N.lib().sq_kmeans_workspace_bytes_bounded if bounded else N.lib().sq_kmeans_workspace_bytes
    need = size(G, num_tokens, num_centroids, 128)
    return torch.empty(need, dtype=torch.uint8, device=device)


def _step(data, centroids, max_idx, normalize_centroids, workspace, state, bounded):
    """One Lloyd step, centroids updated in place; (assignment, cluster sizes)."""
    _require(data, "data")
    batch_size, num_tokens, dim = data.shape
    num_centroids = centroids.shape[1]
    assert num_centroids % 32 == 0
    if max_idx is None:
        max_idx = torch.empty((batch_size, num_tokens), dtype=torch.int32, device=data.device)
    data_cnt = torch.empty((batch_size, num_centroids), dtype=torch.int32, device=data.device)
    if workspace is None:
        workspace = _workspace(batch_size, num_tokens, num_centroids, data.device, bounded)
    b = [N.dl(t) for t in (data, centroids, max_idx, data_cnt, workspace)]
    train = N.lib().sq_kmeans_train_bounded if bounded else N.lib().sq_kmeans_train_stateful
    N.check(train(*[N.ptr(x) for x in b], 1 if normalize_centroids else 0, int(state), N.current_stream(data.device)))
    return max_idx, data_cnt


def _triton_k_means_train(data, centroids, max_idx=None, normalize_centroids=True, return_indices=False,
                          workspace: Optional[torch.Tensor] = None, state: int = N.KMEANS_STATELESS, bounded: bool = False):
    """One Lloyd step, centroids updated in place (kmeans.py:127-196).  With `return_indices` also returns
    the assignment and the largest cluster size (a host sync, like the reference's `.item()`, :195).
    `state` (extension, for a run of steps over the same data with the same `max_idx` and `workspace`):
    `N.KMEANS_KEEP_SUMS` leaves the clusters' exact sums in the workspace, `N.KMEANS_APPLY_CHANGES` forms the new
    centroids from those sums and the tokens that changed cluster instead of re-summing every row (same bits).
    `bounded` (for a whole run, with the workspace of `_workspace(..., bounded=True)`): centroids that cannot win are left out of
    the assignment (`sq_kmeans_train_bounded`, same bits)."""
    max_idx, data_cnt = _step(data, centroids, max_idx, normalize_centroids, workspace, state, bounded)
    if return_indices:
        return centroids, max_idx, int(data_cnt.max().item())
    return centroids


def triton_reverse_index(max_idx, num_centroids: int, max_cluster_size: int, workspace: Optional[torch.Tensor] = None):
    """clusters[g,c,:size] = token ids of cluster c in ascending order (kmeans.py:233-262)."""
    _require(max_idx, "max_idx")
    batch_size, num_tokens = max_idx.shape
    clusters = torch.empty((batch_size, num_centroids, max(int(max_cluster_size), 1)), dtype=torch.int32, device=max_idx.device)
    cluster_size = torch.empty((batch_size, num_centroids), dtype=torch.int32, device=max_idx.device)
    if workspace is None:
        workspace = _workspace(batch_size, num_tokens, num_centroids, max_idx.device)
    b = [N.dl(t) for t in (max_idx, clusters, cluster_size, workspace)]
    N.check(N.lib().sq_reverse_index(*[N.ptr(x) for x in b], N.current_stream(max_idx.device)))
    return clusters, cluster_size


def triton_index_add(value, max_idx, num_centroids: int, workspace: Optional[torch.Tensor] = None):
    """Per-cluster sums of `value`, in value's dtype (kmeans.py:307-329)."""
    _require(value, "value")
    batch_size, num_tokens, dim = value.shape
    out = torch.empty((batch_size, num_centroids, dim), dtype=value.dtype, device=value.device)
    if workspace is None:
        workspace = _workspace(batch_size, num_tokens, num_centroids, value.device)
    b = [N.dl(t) for t in (value, max_idx, out, workspace)]
    N.check(N.lib().sq_index_add(*[N.ptr(x) for x in b], N.current_stream(value.device)))
    return out


FULL_RESUM_STEPS = 3   # Lloyd steps that re-sum every row before the sums are carried (most tokens still move in them)


def _bounded(groups: int, tokens: int, num_centroids: int, carried_steps: int) -> bool:
    """Whether a run's carried steps leave out centroids that cannot win, `tokens` those of one group.  In us: what a step saves on keys
    around C / 2 centres goes with the products left out, less the rows it gathers; its bounds go with the squares of the
    centroids and its launch is there in any case.  Preparing takes some 50 us once, and a run that finds nothing to leave out has lost
    20 us and 2 a step, so that much has to be won.  Not where a step saves next to nothing, however many there are, nor with less than two
    workgroups a CU, whose length is the chain of loads.  Ten steps (seven carried), us without / with around 512 centres of width 0.3, and
    around centres that overlap (width 0.8): 1024 centroids 4 x 131072 tokens 1474 / 1204 (1437 / 1468), 4 x 62000 807 / 745
    (785 / 817), 8 x 34000 970 / 930 (956 / 991), 16 x 28000 1397 / 1345 (1391 / 1432), 2 x 104000 769 / 743 (731 / 763); outside 8 x 33000
    992 / 991 (980 / 1019), 1 x 131072 610 / 649, 16 x 24000 1256 / 1272.  2048 centroids 4 x 65536 1407 / 1230, outside 4 x 33000 1066 / 1072; 512
    centroids 8 x 90000 1199 / 1139, outside 4 x 131072 985 / 961 (947 / 982).  Five steps, 1024 centroids: 4 x 122000 814 / 775 (791 / 813), outside
    4 x 70000 599 / 605.  Forty or fifty: 4 x 131072 tokens, 512 centroids 3694 / 3284, 1024 centroids 8 x 34000 3223 / 2821, 4 x 45000 2109 /
    1997, outside 1 x 131072 1634 / 1778, 4 x 20000 1727 / 2246."""
    rows, c = groups * tokens / 131072, num_centroids / 1024
    saved = (17.5 * c - 5) * rows - 1.4 * groups * c * c - 4
    return 512 <= num_centroids <= 2048 and rows >= 1 and saved >= 7.5 and carried_steps * saved >= 72


def segment_k_means(key, value, num_centroids: int, num_iters: int = 10, num_segments: int = 1):
    """kmeans.py:332-375: strided initial centroids, `num_iters-1` normalised steps on the segmented data,
    one un-normalised step on the whole data, then value sums and the reverse index.

    From the fourth step on the exact cluster sums are carried from step to step and only the tokens that changed
    cluster are re-added (`sq_kmeans_train_stateful`): the same centroids bit for bit, without reading the keys a second
    time per step.  With one segment the final step runs on the same tensors and continues that way."""
    _require(key, "key")
    num_groups, num_tokens, head_dim = key.shape
    centroid_indices = torch.arange(num_centroids, dtype=torch.float32, device=key.device) * (num_tokens / num_centroids)
    centroid_indices += num_tokens / num_centroids / 2
    centroid_indices = centroid_indices.to(torch.int64)
    centroids = torch.index_select(key, dim=1, index=centroid_indices)
    assert num_centroids % num_segments == 0
    num_tokens_per_segment = num_tokens // num_segments
    num_centroids_per_segment = num_centroids // num_segments
    data = key[:, : num_tokens_per_segment * num_segments].reshape((-1, num_tokens_per_segment, head_dim))
    centroids = centroids.reshape((-1, num_centroids_per_segment, head_dim)).contiguous()
    max_idx = torch.empty((data.shape[0], data.shape[1]), dtype=torch.int32, device=data.device)
    one_run = num_segments == 1 and data.shape[1] == num_tokens   # the last step continues on the same tensors
    bounded = _bounded(data.shape[0], data.shape[1], num_centroids_per_segment, num_iters - FULL_RESUM_STEPS - (0 if one_run else 1))
    ws = _workspace(data.shape[0], data.shape[1], num_centroids_per_segment, key.device, bounded)
    carried = False
    for it in range(num_iters - 1):
        state = N.KMEANS_STATELESS if it < FULL_RESUM_STEPS - 1 else (N.KMEANS_APPLY_CHANGES if carried else N.KMEANS_KEEP_SUMS)
        centroids = _triton_k_means_train(data, centroids, max_idx=max_idx, normalize_centroids=True,
                                          return_indices=False, workspace=ws, state=state, bounded=bounded)
        carried = state != N.KMEANS_STATELESS
    if one_run and carried:
        # the same tensors, the same workspace: the last (un-normalised) step continues from the carried sums
        state = N.KMEANS_APPLY_CHANGES
    else:
        data = key.reshape((-1, num_tokens, head_dim))
        centroids = centroids.reshape((-1, num_centroids, head_dim))
        ws = _workspace(num_groups, num_tokens, num_centroids, key.device)
        max_idx, state, bounded = None, N.KMEANS_STATELESS, False
    max_idx, data_cnt = _step(data, centroids, max_idx, False, ws, state, bounded)
    # The host has to know the largest cluster before it can lay out the token table.  The number travels while the value sums run, and
    # the table's launches are there when these end; asked for in front of the sums the GPU waited for the host (4 x 131072 tokens, 1024
    # centroids 1103 -> 1093 us a run, 4 x 70000 800 -> 791, 8 x 33000 944 -> 938).
    largest = torch.empty((), dtype=torch.int32, device="cpu", pin_memory=True).copy_(data_cnt.max(), non_blocking=True)
    known = torch.cuda.Event()
    known.record(torch.cuda.current_stream(key.device))
    value_sum = triton_index_add(value.reshape((-1, num_tokens, head_dim)), max_idx, num_centroids, workspace=ws)
    known.synchronize()
    clusters, cluster_size = triton_reverse_index(max_idx, num_centroids, int(largest), workspace=ws)
    return centroids, value_sum, clusters, cluster_size


def topk_select(query, centroids, clusters, cluster_size, k: int, num_kv_groups: int, out=None, workspace=None):
    """Centroid-scored token selection (no reference counterpart): query [B,Hq,D] -> token ids int32 [G,k].
    `out` (int32 [G,k], contiguous) and `workspace` (`_workspace(G, 1, C, device)`) may be passed by a caller that
    selects every step."""
    _require(query, "query")
    res = N.host_calls().topk_select(query, centroids, clusters, cluster_size, k, num_kv_groups, out, workspace, N.current_stream(query.device))
    if res is not None:
        return N.result(res)
    G, C, _ = centroids.shape
    if out is None:
        out = torch.empty((G, k), dtype=torch.int32, device=query.device)
    ws = workspace if workspace is not None else _workspace(G, 1, C, query.device)
    ptrs, held = N.borrow(query, centroids, clusters, cluster_size, out, ws)
    N.check(N.lib().sq_topk_select(*ptrs, num_kv_groups, N.current_stream(query.device)))
    return out


def cluster_order(clusters: torch.Tensor, cluster_size: torch.Tensor):
    """From the reverse index (`clusters` int32 [G,C,M], `cluster_size` int32 [G,C]) the two tables of a cache kept in
    cluster order (no reference counterpart): `order` int32 [G,n] lists every group's tokens cluster by cluster (n = the
    largest group total; shorter groups are padded with -1), and `positions` int32 [G,C,M] holds, in the layout of
    `clusters`, where each of those tokens sits in that list.  `topk_select(query, centroids, positions, cluster_size,
    ...)` then yields rows of the reordered cache instead of token ids."""
    G, C, M = clusters.shape
    size = cluster_size.to(torch.int64)
    offset = torch.cumsum(size, dim=1) - size                                   # [G,C] exclusive prefix
    slot = torch.arange(M, device=clusters.device).view(1, 1, M)
    used = slot < size.unsqueeze(-1)                                            # [G,C,M]
    positions = torch.where(used, offset.unsqueeze(-1) + slot, torch.zeros_like(slot)).to(torch.int32)
    n = int(size.sum(dim=1).max().item())
    order = torch.full((G, n), -1, dtype=torch.int32, device=clusters.device)
    rows = torch.arange(G, device=clusters.device).view(G, 1, 1).expand(G, C, M)
    order[rows[used], positions[used].long()] = clusters[used]
    return order, positions


def reorder_cache(key_cache: torch.Tensor, value_cache: torch.Tensor, order: torch.Tensor):
    """Copies of a layer's cache [B,L,Hkv,D] with each kv head's rows in the order `order` int32 [B*Hkv,n] gives
    (`sq_kv_cache_reorder`): out[b, p, h] = cache[b, order[b*Hkv + h, p], h]; rows for -1 are zero."""
    _require(key_cache, "key_cache")
    _require(value_cache, "value_cache")
    B, _, H, D = key_cache.shape
    n = order.shape[1]
    key_out = torch.empty((B, n, H, D), dtype=key_cache.dtype, device=key_cache.device)
    value_out = torch.empty_like(key_out)
    b = [N.dl(t) for t in (key_cache, value_cache, order, key_out, value_out)]
    N.check(N.lib().sq_kv_cache_reorder(*[N.ptr(x) for x in b], N.current_stream(key_cache.device)))
    return key_out, value_out

