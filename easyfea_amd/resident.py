"""Plans of the resident solves (``efea_solve_resident``): which block of the
chip owns which nodes, where each neighbour's value lies (in the block's own
LDS or its halo) and which nodes' values other blocks read.

A plan belongs to a sparsity pattern and, for two-level solves, its
aggregates; it is built once and kept with them.  With aggregates the blocks
take runs of 64 / lanes nodes (chunks) of one aggregate each, in aggregate
order; without, the nodes are bisected along coordinates into one part per
block.
"""

from __future__ import annotations

import ctypes as C
import heapq
from typing import Optional

import numpy as np
import torch

from . import _lib

WAVES = 8  # of a block of 512 threads
COLLECTORS = 256  # threads of a block that collect the restriction


def shape(dof_n: int, max_neighbours: int, min_passes: int) -> Optional[tuple]:
    """(lanes per node, slots per lane, passes) of the smallest kernel variant, or None."""
    v = [C.c_int(), C.c_int(), C.c_int()]
    ok = _lib.call("efea_resident_shape", dof_n, max_neighbours, min_passes, *[C.byref(c) for c in v])
    return tuple(c.value for c in v) if ok else None


def bisect(coord: np.ndarray, parts: int) -> list:
    """The nodes in ``parts`` compact groups of nearly equal size (recursive
    coordinate bisection), each in increasing order."""
    c = np.zeros((coord.shape[0], 3))
    c[:, :coord.shape[1]] = coord  # of one to three columns
    order, ptr_ = np.empty(c.shape[0], dtype=np.int32), np.empty(parts + 1, dtype=np.int32)
    _lib.call("efea_resident_bisect", c.shape[0], c.ctypes.data, parts, order.ctypes.data, ptr_.ctypes.data)
    return np.split(order, ptr_[1:-1])


def block_count(least: int, per_block: int, max_blocks: int, agg: np.ndarray, nc: int) -> int:
    """Number of blocks for chunks of the aggregates ``agg`` (in order).  More
    blocks than the nodes need cost time in the exchange (about 25 cycles a
    block and iteration), more pieces in a block its rows of the coarse inverse
    (about 1.3 cycles per column and piece): measured, 300 x 300 QUAD4 (nc
    1,536) 32,000 cycles an iteration with 192 blocks of up to four pieces,
    24,800 with 256 of two; notched 200 x 200 (nc 768) 19,600 with 161 of three,
    20,800 with 256 of two; 360 x 39 (nc 192) 14,000 with 64 of one, 15,700
    with 256."""
    best = None
    n = agg.size
    for nblk in range(least, min(max_blocks, n) + 1):
        block = np.arange(n) * nblk // n
        if np.bincount(block).max() > per_block:
            continue
        new = np.append(True, (agg[1:] != agg[:-1]) | (block[1:] != block[:-1]))
        cost = 25 * nblk + 1.3 * nc * np.bincount(block[new]).max()
        if best is None or cost < best[0]:
            best = (cost, nblk)
    return best[1]


def layout(coord: Optional[np.ndarray], Nn: int, dof_n: int, max_neighbours: int, max_blocks: int, ag=None):
    """(lanes, slots, passes, rows, chunk_agg): ``rows`` (blocks, positions) holds
    the node of each position (-1: none), ``chunk_agg`` (blocks, chunks) the
    aggregate of each chunk (-1: none; absent without aggregates).  None when
    the nodes do not fit ``max_blocks`` blocks of any kernel variant."""
    passes = 0
    while True:
        v = shape(dof_n, max_neighbours, passes + 1)
        if v is None:
            return None
        lanes, slots, passes = v
        per, per_block = 64 // lanes, WAVES * passes
        nloc = per * per_block
        if ag is None:
            nblk = -(-Nn // nloc)
        else:
            chunks = -(-np.diff(ag.agg_ptr).astype(np.int64) // per)
            nblk = -(-int(chunks.sum()) // per_block)
        if nblk <= max_blocks:
            break
    rows = np.full((nblk, nloc), -1, dtype=np.int32)
    if ag is None:
        if coord is None:
            return None
        for b, ids in enumerate(bisect(coord, nblk)):
            rows[b, :ids.size] = ids
        return lanes, slots, passes, rows, None
    n = int(chunks.sum())
    agg = np.repeat(np.arange(ag.nagg), chunks)              # aggregate of each chunk
    nblk = block_count(nblk, per_block, max_blocks, agg, ag.nagg * (3 if lanes == 2 else 6))
    rows = np.full((nblk, nloc), -1, dtype=np.int32)
    within = np.arange(n) - np.repeat(np.cumsum(chunks) - chunks, chunks)
    block = np.arange(n) * nblk // n                          # even runs of chunks
    local = np.arange(n) - np.searchsorted(block, np.arange(nblk))[block]
    pos = ag.agg_ptr[agg][:, None] + within[:, None] * per + np.arange(per)[None, :]
    have = pos < ag.agg_ptr[agg + 1][:, None]
    nodes = np.where(have, ag.agg_nodes[np.minimum(pos, Nn - 1)], -1)
    rows.reshape(nblk, per_block, per)[block, local] = nodes
    chunk_agg = np.full((nblk, per_block), -1, dtype=np.int64)
    chunk_agg[block, local] = agg
    return lanes, slots, passes, rows, chunk_agg


def pieces(chunk_agg: np.ndarray) -> dict:
    """The runs of one block's chunks of one aggregate, numbered through
    (``piece_chunk``: each one's first and past-last chunk, for checks of a plan)."""
    nblk, nch = chunk_agg.shape
    new = chunk_agg >= 0
    new[:, 1:] &= chunk_agg[:, 1:] != chunk_agg[:, :-1]
    blk, first = np.nonzero(new)
    agg = chunk_agg[blk, first]
    ptr = np.searchsorted(blk, np.arange(nblk + 1))
    used = (chunk_agg >= 0).sum(1)
    last = np.append(first[1:], 0)
    end = np.append(blk[1:], -1) != blk
    last[end] = used[blk[end]]
    cp = np.where(chunk_agg >= 0, np.cumsum(new, 1) - 1, -1)
    return dict(piece_ptr=ptr, piece_agg=agg, piece_chunk=np.stack([first, last], 1).ravel(),
                chunk_piece=cp.ravel(), max_pieces=int(np.diff(ptr).max()))


def collection(nm: int, nagg: int, pc: dict) -> np.ndarray:
    """(entries, COLLECTORS): what each thread collects of the published
    restrictions, as ``include/efea.h`` describes it; the components (their
    pieces stay together) are dealt to the threads, largest first, to the least
    loaded."""
    nblk = len(pc["piece_ptr"]) - 1
    line = -(-(3 + nm * pc["max_pieces"]) // 8) * 8
    blk = np.repeat(np.arange(nblk), np.diff(pc["piece_ptr"]))
    place = blk * line + 3 + nm * (np.arange(blk.size) - pc["piece_ptr"][blk])
    first = np.searchsorted(pc["piece_agg"], np.arange(nagg + 1))
    groups = [(a * nm + m, place[first[a]:first[a + 1]] + m) for a in range(nagg) for m in range(nm)]
    groups.sort(key=lambda gr: -len(gr[1]))  # stable: neighbouring components stay together
    lists = [[] for _ in range(COLLECTORS)]
    heap = [(0, t) for t in range(COLLECTORS)]
    for dest, offs in groups:
        load, t = heapq.heappop(heap)
        lists[t] += [int(o) | dest << 16 | (1 << 31 if i == len(offs) - 1 else 0) for i, o in enumerate(offs)]
        heapq.heappush(heap, (load + len(offs), t))
    out = np.full((max(len(v) for v in lists), COLLECTORS), -1, dtype=np.int64)
    for t, v in enumerate(lists):
        out[:len(v), t] = v
    return np.where(out >= 1 << 31, out - (1 << 32), out).astype(np.int32)


def neighbours(rows: torch.Tensor, node_ptr: torch.Tensor, node_cols: torch.Tensor, lanes: int, slots: int,
               passes: int) -> dict:
    """Halo lists, exchange numbers and the local neighbour positions of a
    layout, as ``include/efea.h`` describes them, on the host."""
    nblk, nloc = rows.shape
    kept = slots - 1 if lanes == 1 else slots  # a scalar row's own node has no entry
    rows, node_ptr, node_cols = (t.to("cpu", torch.int32).contiguous() for t in (rows, node_ptr, node_cols))
    i32 = dict(dtype=torch.int32)
    out = dict(lidx=torch.empty(nblk * passes * kept * 64 * WAVES, dtype=torch.int16),
               halo_ptr=torch.empty(nblk + 1, **i32), halo_ex=torch.empty(node_cols.numel(), **i32),
               pub=torch.empty(nblk * nloc, **i32), pub_ptr=torch.empty(nblk + 1, **i32),
               pub_pos=torch.empty(nblk * nloc, **i32), self=torch.empty(nblk * nloc, **i32))
    nex, max_halo = C.c_int(), C.c_int()
    _lib.call("efea_resident_neighbours", node_ptr.numel() - 1, node_ptr.data_ptr(), node_cols.data_ptr(), lanes,
              slots, passes, nblk, rows.data_ptr(), out["lidx"].data_ptr(), out["halo_ptr"].data_ptr(),
              out["halo_ex"].data_ptr(), out["halo_ex"].numel(), *[out[n].data_ptr() for n in (
                  "pub", "pub_ptr", "pub_pos", "self")], C.addressof(nex), C.addressof(max_halo))
    return dict(out, halo_ex=out["halo_ex"][:int(out["halo_ptr"][-1])], pub_pos=out["pub_pos"][:nex.value],
                nex=nex.value, max_halo=max_halo.value)


class Resident:
    """The device plan of a pattern (and its coarse space ``cs``)."""

    def __init__(self, plan: _lib.ResidentPlan, keep: dict, Nn: int):
        self.plan, self._keep = plan, keep
        self.nbytes = int(_lib.load().efea_resident_workspace_bytes(Nn, C.byref(plan)))

    @staticmethod
    def build(pattern, cs=None) -> Optional["Resident"]:
        """None when no kernel variant takes the pattern."""
        if cs is not None and pattern.dof_n == 1:
            return None
        cus = torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count
        lay = layout(pattern.coord, pattern.Nn, pattern.dof_n, pattern.host.max_neighbours, cus,
                     None if cs is None else cs.ag)
        if lay is None:
            return None
        lanes, slots, passes, rows, chunk_agg = lay
        if rows.shape[1] + pattern.Nn > 2**31 - 1:
            return None
        h = pattern.host
        nb = neighbours(torch.from_numpy(rows), torch.from_numpy(h.node_ptr), torch.from_numpy(h.node_cols), lanes,
                        slots, passes)
        rows_dev = torch.from_numpy(rows).to("cuda")
        keep = dict(rows=rows_dev, **{n: nb[n].to("cuda") for n in ("lidx", "halo_ptr", "halo_ex", "pub", "pub_ptr",
                                                                    "pub_pos", "self")})
        pl = _lib.ResidentPlan(dof_n=pattern.dof_n, slots=slots, passes=passes, nblk=rows.shape[0],
                               max_halo=nb["max_halo"], nex=nb["nex"])
        if rows.shape[1] + nb["max_halo"] > 65535:
            return None
        if cs is not None:
            pc = pieces(chunk_agg)
            pl.nagg, pl.npiece, pl.max_pieces = cs.nagg, pc["piece_agg"].size, pc["max_pieces"]
            pc["collect"] = collection(cs.nm, cs.nagg, pc)
            pl.ncollect = pc["collect"].shape[0]
            for n in ("piece_ptr", "piece_agg", "chunk_piece", "collect"):
                keep[n] = torch.from_numpy(pc[n].astype(np.int32)).to("cuda")
        for n, t in keep.items():
            setattr(pl, n, t.data_ptr() if t.numel() else rows_dev.data_ptr())  # never null
        if not _lib.load().efea_resident_fits(C.byref(pl)):
            return None
        return Resident(pl, keep, pattern.Nn)
