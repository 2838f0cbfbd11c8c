"""Host driver of the HIP cost engine: holds a packed problem in HBM and runs
the kernels through the C ABI.  PyTorch is used only for device memory and the
current HIP stream."""
from __future__ import annotations

import ctypes as C
import threading
import weakref
from typing import Dict, Optional

import numpy as np
import torch

from . import _lib
from .packed import CHUNK_SHIFT, ITEM_ENTRIES, MAX_MESH_DIMS, PackedGraph

_LARGE_BLOCKS_FROM = 8192  # mean entries per edge block
_UPLOAD_ARENA_BYTES = 8 << 20  # descriptor arrays of one problem that go up in one copy
_UPLOAD_ARENA_MAX_ARRAY = 2 << 20
_SCORE_LANES_FROM = 32768  # assignments: below, always with the terms side by side (from the table or the arrays)
_SCORE_FROM_TABLE = True  # the three ways of scoring a graph with large blocks can be switched off (tests do)
_SCORE_COMPACT = True
_SCORE_SMALL_FROM_TABLE = True
_SCORE_FROM_TILES = True  # small blocks: matrices through LDS by tiles, while the table stands for the arrays
_SCORE_TERMS_ABOVE = True  # from _SCORE_LANES_FROM on, too, up to the lines below (tests switch them off)
# Where a graph with small blocks has no tiles, the terms of so many assignments gathered side by side are faster than a
# walk over records with a lane per assignment, which takes as long for one as for 2^18 of them.  In ms, terms and records,
# random at 114 688, 131 072 and 139 264, explicit at 131 072, 163 840 and 172 032: random DAG of 1 200 nodes with up to 150
# strategies 1.16, 1.43 and 1.42, 1.43 and 1.51, 1.42, and 1.58, 2.26 and 2.22, 2.29 and 2.34, 2.30; of 300 nodes on 4x8x8
# 0.30, 0.38 and 0.32, 0.38 and 0.34, 0.37, and 0.36, 0.44 and 0.43, 0.45 and 0.45, 0.45.  Graphs whose terms hit the caches
# more often would gain above, too (Llama-3-8B graph, compressed table, 196 608 5.3, 7.2), but those have tiles.
_SCORE_TERMS_UP_TO_RECORDS = {"random": 131072, "explicit": 163840}
# The same where the walk is one over tile images, which is as long for one assignment as for the 65 536 that are a
# wavefront a SIMD; terms go in rounds of 16 384.  In ms, terms and images: Llama-3-8B graph, random, at 114 688 and 131 072
# 2.49, 2.90 and 2.80, 2.91, explicit, at 81 920 and 90 112 2.48, 2.70 and 3.16, 2.70; 12-layer GPT-2 graph 0.77, 0.81 and
# 0.86, 0.81, and 0.64, 0.72 and 0.81, 0.72.
_SCORE_TERMS_UP_TO_IMAGES = {"random": 114688, "explicit": 81920}
# Random assignments that carry no sums: from images of finished entries beyond these many, the second where a tile has
# room for few argument rows of the graph's mean size, so that its beginning counts.  In ms, finished entries, tile images (from 262 144 on lanes of
# several), terms: 12-layer GPT-2 graph (173 rows), 90 112 0.62, 0.81, 0.66, 131 072 0.64, 0.81, 0.87, 262 144 0.98,
# 1.22, 2^20 2.24, 3.42; Llama-3-8B graph (5.1), 131 072 2.98, 2.91, 2.80, 163 840 3.31, 3.65, 3.45, 262 144 3.68, 4.68,
# 2^20 7.24, 10.41; MoE graph (6.0), 131 072 1.59, 1.57, 1.53.
_SCORE_PAIRS = True
_SCORE_PAIRS_FROM, _SCORE_PAIRS_ROWS = (81920, 131072), 8
# Not where a graph is a few tiles, which the walks without images in front go through meanwhile.  In us, finished entries,
# tile images and lanes of several, at 131 072, 262 144 and 2^20: random DAG of 39 edges (5 tiles of finished entries, 3 of
# images) 28.6, 23.2, 28.1 and 35.0, 30.5, 29.5 and 64.1, 94.9, 56.4, of 61, 524 288 55.2 and, lanes of several, 51.5, of 84
# (11, 8) 40.2, 39.1, 51.0 and 51.9, 56.8, 51.6 and 103, 200, 116.  Explicit ones beyond 2^18, tile images and lanes of several,
# 524 288 and 2^20: 39 edges 52.2, 43.6 and 92.4, 83.7, 84 (8 tiles) 94.7, 85.0 and 177, 168, 138 (13) 138, 138.  And explicit
# ones up to 114 688 go by their terms where a tile has few edges: 100-node DAG of 10 to 60 strategies (3.4), 98 304 98 and 67.
_SCORE_PAIRS_TILES, _SCORE_IMAGES_TILES, _SCORE_IMAGES_EDGES = 10, 12, 4
# Else, random assignments up to which tile images are walked with a lane each; beyond, lanes take two or four, which
# share a tile's draws of far producers and unpacking.  In ms, images and lanes of several, at 196 608 and 262 144:
# Llama-3-8B graph 3.65, 4.59 and 4.48, 4.68; 12-layer GPT-2 graph 1.06, 1.31 and 1.31, 1.21.  Explicit ones at any number: at
# 131 072, 262 144, 524 288 and 2^20 of the Llama-3-8B graph 2.6, 3.8, 7.5, 14.9 against 5.7, 6.7, 8.5, 17.0.
_SCORE_IMAGES_UP_TO = 196608
_SCORE_STREAM = True  # random assignments on graphs with large blocks: matrices as a stream of pieces through LDS
_SCORE_TERM_RECORDS = True  # terms side by side from records of the edges and nodes, made in front of them
# But not where a graph is a few of the smallest batches' tiles: there the records' own launch costs more than it saves.
# Up to so many (assignments; edges or nodes on graphs with small blocks; with large ones, whose entries a workgroup waits
# for longer in the form without records) it is one launch.  In us, a call among others, from records and without: small
# blocks, 1-layer GPT-2 graph (318 edges), random, 100 and 2 048 assignments 15.6, 10.6 and 15.6, 12.9; 2 layers (552), 1 024 and
# 1 500 15.5, 14.2 and 15.4, 16.3; 3 layers (786), 600 and 1 024 15.7, 16.0 and 15.8, 16.8; 4 layers (1 020), 256 17.8, 17.4;
# 5-layer Llama-3-8B graph (1 378), 100 19.9, 20.8.  Large blocks, 1-layer 70B decoder (318), 100, 1 024 and 1 500 15.6, 10.5
# and 15.5, 14.8 and 16.0, 18.2; windows of the planner DAG of 60 nodes (102), 100 and 2 048 34.2, 30.4 and 34.5, 33.3, of 140
# (255), 600 and 1 024 35.3, 34.9 and 36.2, 37.2, of 300 (559), 256 38.2, 40.0.
# Of the smallest graphs larger batches, too: random DAG of 11 edges, 32 768 and 65 536 13.7, 9.6 and 15.6, 12.3, of 39, 5 000,
# 16 384 and 32 768 14.0, 11.5 and 14.0, 9.7 and 14.0, 11.2, of 61, 32 768 16.2, 13.6, of 84, 16 384 and 32 768 14.1, 12.1 and
# 13.9, 17.6, of 138, 5 000 15.2, 16.7; large blocks, 39, 5 000 and 16 384 13.7, 11.9 and 13.6, 10.0.
_SCORE_TERM_FIELDS_UP_TO = ((256, 1152, 512), (640, 640, 320), (1024, 640, 192), (2048, 384, 192), (16384, 96, 96), (32768, 64, 48),
                               (65536, 16, 16))
# Matrices of up to this many LDS tiles (64 KB each) go through LDS in the table scorer, larger
# ones are read in place.  Measured on a 3 000-node window of the stress DAG, 2^20 assignments:
# 17.9 ms with 1, 17.4 with 2, 18.0 with 4, 18.35 with 8 or 16.  (A lower bound, small matrices
# read in place to save their barrier, only cost time: 17.4 -> 18.9 ms at 1 024 doubles.)
_SCORE_STAGE_TILES = 2
# The table scorers take as long whatever the batch, 0.85 us a piece of a matrix (random assignments) or 2.5 us an
# edge (explicit ones), terms side by side about 9 ns (random) and 12 per edge and 1 000 assignments.  In ms, random ones,
# terms and table: window of the planner DAG (1.6 pieces an edge), 131 072 and 147 456 assignments 3.64, 4.08 and 4.43, 4.15;
# 8-layer 70B decoder on 2x2x4 (2.6 pieces), 131 072 2.09, 4.52.  Explicit ones, that window, 163 840 and 196 608 6.03,
# 7.89 and 7.76, 7.89.  Random ones without a list of pieces (more than 819 strategies; not made before a graph is
# recorded) go through the table edge by edge, 1.75 us each: that window, 155 648, 163 840 and 172 032 4.28, 5.05 and 4.59, 5.03
# and 4.98, 5.04, 120 nodes of 830 to 900 strategies, 147 456 and 163 840 0.33, 0.36 and 0.37, 0.36, 60 of 1 030 to 1 100, 163 840
# and 180 224 0.21, 0.22 and 0.23, 0.22.  The table it is from this many assignments on, times pieces per edge over 1.5
# (random), or 1.25 (without pieces), or 1.5 (explicit).
_SCORE_TABLE_FROM = 131072
_SCORE_TABLE_PIECES, _SCORE_TABLE_EDGES, _SCORE_TABLE_EXPLICIT = 1.5, 1.25, 1.5
# But random ones edge by edge where many matrices are more than two tiles: the stream copies every piece of them to each CU,
# edge by edge they are read in place, an entry a draw, which is little while few assignments share them.  What an edge
# takes, us: as a stream, a piece and, at 2^20 assignments, the draws on top; edge by edge, at least, a tile, a matrix in
# place, and on top at 2^20, in all, for a matrix in place, and, by the square, where nearly all are (no copies then keep
# the CUs at the same matrix).  Terms, ns for an edge and 1 000 assignments: at least, with a
# matrix, and for each MB of the block table, at most so much.  In ms, terms, stream and edge by edge, at 131 072, 262 144, 524 288
# and 2^20: 2-layer 70B decoder on 2x2x4 (2.9 pieces an edge, 0.41 in place, 21 MB) 0.56, 1.51, 0.97 and 1.13, 1.58, 0.97 and
# 2.34, 1.76, 1.26 and 4.76, 2.16, 1.88; 8 layers of it, compressed (2.3, 0.25, 16 MB) 2.06, 4.53, 3.99 and 4.03, 4.77, 3.99 and
# 8.01, 5.38, 4.98 and 16.0, 6.74, 7.18; 300-node DAG, not compressed, 140 to 170 strategies (3.4, 1.0, 79 MB) 0.63, 1.33, 0.65 and
# 1.43, 1.40, 0.64 and 3.06, 1.53, 1.26 and 6.35, 1.84, 3.59 (786 432: 4.71, 1.70, 2.66); 95 to 110 (2.0, 0, 35 MB) 0.48, 0.70,
# 0.98 and 1.17, 0.75, 1.00 and 2.65, 0.88, 1.12 and 5.63, 1.16, 1.38; compressed, 250 to 300 (1.8, 0.24, 23 MB) 0.35, 0.47, 0.54 and 0.70, 0.50, 0.55 and
# 1.44, 0.58, 0.68 and 2.94, 0.75, 0.98; 400-node window of the planner DAG, not compressed (5.1, 0.41, 429 MB) 1.68, 9.83, 2.52
# and 3.65, 9.90, 2.51 and 7.87, 10.2, 3.42 and 16.3, 11.1, 5.42.
_SCORE_STREAM_US, _SCORE_TABLE_US = (0.92, 1.15), (1.05, 0.7, 0.85, 1.1, 1.7, 3.5)
_SCORE_TERMS_NS = (2.2, 4.5, 0.05, 8.0)
_SCORE_PER_LANE = 0  # assignments per lane of the compact scorer; 0: the library chooses
# Assignments from which one lane each beats several wavefronts per 64 assignments, by the number
# of wavefronts.  Lanes go in rounds of 2^18 that cost the same however full, wavefronts by the
# assignment, so that near the end of a round the lanes win: from seven eighths of the second round (of the
# first, with sixteen) on.  In ms, wavefronts and lanes: two, at 400 000 and 524 288 assignments, 12-layer GPT-2
# graph 4.74, 5.93 and 6.02, 6.02, 4-layer 70B decoder on 4x8x8 2.65, 3.22 and 3.36, 3.22, Llama-3-8B graph 13.7,
# 20.2 and 17.5, 21.2; at 1 048 575 12.2, 11.1 and 6.49, 5.99 and 35.5, 35.4.  Sixteen, at 220 000 and 262 143,
# window of the planner DAG of 1 600 nodes 5.49, 6.33 and 6.34, 6.30, of 60 nodes 0.242, 0.260 and 0.270, 0.262.
_SAMPLE_LANES_FROM = {2: 458752, 16: 229376}
_SAMPLE_WAVES = 0  # 2 or 16: tests
# Graphs of at most 64 strategies a node: by tiles of nodes through LDS.  In ms, tiles, and wavefronts
# or lanes: Llama-3-8B graph, 100, 131 072 and 524 288 assignments 2.0, 2.4, 7.2 and 3.0, 5.1, 21.2; 12-layer GPT-2 graph,
# 100 and 131 072 0.66, 0.86 and 0.91, 1.56.
_SAMPLE_TILES = True
# But not small batches on graphs with work for sixteen wavefronts: tiles go node by node, wavefronts by the depth of
# the graph.  What each takes, us: tiles, in all, per node and per tile; a step, in all and per argument row of the mean
# node, for every 16 384 assignments (a workgroup of 64 on each CU).  In us, tiles and wavefronts at 16 384, 32 768, 49 152
# and 65 536: random DAG of 800 nodes (1.4 rows a node, 52 steps) 298, 312, 302, 306 and 102, 177, 254, 328, of 60 nodes
# 55, 56, 56, 56 and 35, 45, 55, 65, of 4 000 1 394, 1 456, 1 402, 1 408 and 409, 779, 1 152, 1 527; 800 nodes of six rows
# 802, 792, 780, 782 and 247, 466, 685, 906, and of one, producers up to 20 back (81 steps), 264, 277, 268, 270 and 126, 222,
# 325, 407.  The rule takes the shorter one at each of these.
_SAMPLE_TILES_US, _SAMPLE_STEP_US = (24.0, 0.16, 3.0), (1.0, 0.3)
# Nor on the smallest graphs, where two wavefronts have few steps.  In all and a step, and the assignments up to which that
# holds (beyond, it grows with them).  In us, among others, tiles and two wavefronts, 16 384, 65 536, 131 072 and 196 608: random
# DAG of 30 nodes (16 steps) 25.6, 17.6 and 26.5, 18.6 and 30.2, 25.0 and 32.5, 37.3, of 60 33.7, 29.7 and 35.4, 31.2 and 40.7,
# 44.0 and 47.0, 67.5, of 100 46.8, 45.8 and 49.6, 48.2; 1-layer GPT-2 graph (243 nodes, 122 steps) 88.5, 101.4.
_SAMPLE_TWO_US, _SAMPLE_TWO_UP_TO = (13.0, 0.85), 100000
# Layouts of a kind (by first_node) an engine makes.  They stay until the engine goes, since a launch on
# another stream or in a graph may still read one; calls beyond take the route that needs none.
_LAYOUTS_KEPT = 16
_READBACK_PINNED = True  # results() copies into pinned host memory (else pageable)
_LUT_TABLE_FROM = 2048  # table units: larger tables are built tile by tile with per-source terms in LDS


def xgmi_config_struct(cfg) -> _lib.ApcXgmiConfig:
    """apc_xgmi_config from any object with XGMITopoConfig's fields."""
    if isinstance(cfg, _lib.ApcXgmiConfig):
        return cfg
    c = _lib.ApcXgmiConfig()
    c.gpus_per_node, c.links_per_gpu = int(cfg.gpus_per_node), int(cfg.links_per_gpu)
    c.link_gbps, c.nic_gbps = float(cfg.link_gbps), float(cfg.nic_gbps)
    c.lat_intra_us, c.lat_inter_us = float(cfg.lat_intra_us), float(cfg.lat_inter_us)
    return c


def score_tile_room(g: PackedGraph):
    """(steps and tiles, units) that apc_score_tiles may need room for: a step per argument row, and per node without
    one; a unit per 32 elements of a step's matrix, and of its node's terms, which every tile that the node goes on in
    places again."""
    rows = np.maximum(np.diff(g.node_edge_off), 1).astype(np.int64)
    units = ((g.edge_sdst.astype(np.int64) * g.edge_ssrc + 31) // 32).sum() + (rows * ((g.node_nstrat + 31) // 32)).sum()
    return g.num_nodes + g.num_edges, max(int(units), 1)


def matrix_sizes(g: PackedGraph, compressed: bool) -> np.ndarray:
    """int64[num_edges]: elements of an edge's matrix in the block table, of distinct words where it is compressed; 0
    where it has none."""
    _, block_off, _, table_off, usrc, udst = g.block_table(compressed)
    size = g.edge_ssrc.astype(np.int64) * g.edge_sdst
    squeezed = (table_off >= 0) & (usrc > 0)
    if squeezed.any():
        block = np.searchsorted(block_off, table_off[squeezed], side="right") - 1
        size[squeezed] = usrc[squeezed].astype(np.int64) * udst[block]
    size[table_off < 0] = 0
    return size


def piece_counts(g: PackedGraph, size: np.ndarray, first_node: int):
    """(pieces, items) of the list apc_score_pieces makes for the walk from ``first_node`` on over matrices of
    ``size`` elements (matrix_sizes), or None where it makes none: what the choice of a scorer needs to know of it."""
    if first_node >= g.num_nodes or size.max(initial=0) > 0x7FFFFFFF - _lib.SCORE_PIECE:
        return None
    first_edge = int(g.node_edge_off[first_node])
    nstrat, ssrc = g.node_nstrat[first_node:], g.edge_ssrc[first_edge:]
    most = 10 * int(nstrat.max()), 2 * int(ssrc.max(initial=0))
    if max(most) > _lib.SCORE_SIDE_BYTES or (sum(most) > _lib.SCORE_SIDE_BYTES and int(
            (10 * nstrat[g.edge_node[first_edge:] - first_node] + 2 * ssrc).max(initial=0)) > _lib.SCORE_SIDE_BYTES):
        return None
    # an edge without a matrix is one piece, too, as is a node without an argument row
    pieces = np.maximum(size[first_edge:] + (_lib.SCORE_PIECE - 1), _lib.SCORE_PIECE) // _lib.SCORE_PIECE
    bare = int((np.diff(g.node_edge_off[first_node:]) == 0).sum())
    return int(pieces.sum()) + bare, len(pieces) + bare


def large_block_costs(counts, size: np.ndarray, tile: int, table_mb: float):
    """What an edge of the walk takes by the three ways of scoring random assignments on large blocks, up to 2^18 and
    what a batch of 2^20 adds (lanes take several): ((stream, on top), (edge by edge, on top, and by the square)), us, and the
    terms, ns for 1 000 of them.  ``counts``: piece_counts; ``size``: matrix_sizes of the walk's edges; ``tile``: elements of
    an LDS tile."""
    n_piece, n_item = counts
    staged = size <= _SCORE_STAGE_TILES * tile
    tiles = int((-(-size[staged] // tile)).sum()) / n_item
    matrices, in_place = int((size > 0).sum()) / n_item, int((~staged).sum()) / n_item
    least, per_tile, per_in_place, top, top_in_place, top_all_in_place = _SCORE_TABLE_US
    terms, per_matrix, per_mb, most_mb = _SCORE_TERMS_NS
    return ((_SCORE_STREAM_US[0] * n_piece / n_item, _SCORE_STREAM_US[1]),
            (least + per_tile * tiles + per_in_place * in_place, top + top_in_place * in_place,
             top_all_in_place if in_place > 0.9 * matrices else 0.0),
            terms + matrices * (per_matrix + min(most_mb, per_mb * table_mb)))


def make_model(mesh_shape, devices_per_host: int, device_name: str, order_mode: int = 0,
               topo_config=None) -> _lib.ApcModel:
    """Cost-model constants for a mesh on a named device (raises ApcError for a
    device the reference's table does not know either).  ``topo_config``: an
    XGMITopoConfig whose link constants replace the reference's NVLink-era ones
    (then ``devices_per_host`` is not used)."""
    lib = _lib.load()
    m = _lib.ApcModel()
    nd = len(mesh_shape)
    assert 1 <= nd <= MAX_MESH_DIMS
    m.ndim = nd
    m.order_mode = int(order_mode)
    shape = (C.c_int32 * MAX_MESH_DIMS)(*([int(x) for x in mesh_shape] + [1] * (MAX_MESH_DIMS - nd)))
    m.mesh_shape = shape
    bw = (C.c_double * MAX_MESH_DIMS)()
    lat = (C.c_double * MAX_MESH_DIMS)()
    _lib.check(
        lib.apc_mesh_topology(C.addressof(shape), nd, int(devices_per_host), C.addressof(bw), C.addressof(lat)),
        "apc_mesh_topology",
    )
    if topo_config is not None:
        a2a = (C.c_double * MAX_MESH_DIMS)()
        xc = xgmi_config_struct(topo_config)
        _lib.check(
            lib.apc_xgmi_topology(C.byref(xc), C.addressof(shape), nd, C.addressof(bw), C.addressof(lat),
                                  C.addressof(a2a)),
            "apc_xgmi_topology")
        m.mesh_a2a_bw = a2a
    m.mesh_bw = bw
    m.mesh_lat = lat
    _lib.check(lib.apc_device_limits(device_name.encode(), C.byref(m)), "apc_device_limits")
    return m


def nccl_config_struct(cfg) -> _lib.ApcNcclConfig:
    """apc_nccl_config from any object with NCCLTopoConfig's fields
    (autoparallel/cost_models/nccl_cost_model.py:67-82); ``arch`` may be an
    int or an enum with an int ``value``."""
    if isinstance(cfg, _lib.ApcNcclConfig):
        return cfg
    c = _lib.ApcNcclConfig()
    c.arch = int(getattr(cfg.arch, "value", cfg.arch))
    c.num_nodes = int(cfg.num_nodes)
    c.gpus_per_node = int(cfg.gpus_per_node)
    c.num_channels = int(cfg.num_channels) if cfg.num_channels is not None else 0
    c.has_nvswitch = int(bool(cfg.has_nvswitch))
    c.has_collnet = int(bool(cfg.has_collnet))
    c.bw_intra = float(cfg.bw_intra)
    c.bw_inter = float(cfg.bw_inter)
    c.net_latency = float(cfg.net_latency)
    return c


def build_nccl_plan(cfg, mesh_shape) -> _lib.ApcNcclPlan:
    """Host plan of the NCCL-tuning model for a mesh (apc_nccl_plan_build)."""
    lib = _lib.load()
    nd = len(mesh_shape)
    shape = (C.c_int32 * MAX_MESH_DIMS)(*([int(x) for x in mesh_shape] + [1] * (MAX_MESH_DIMS - nd)))
    plan = _lib.ApcNcclPlan()
    c = nccl_config_struct(cfg)
    _lib.check(lib.apc_nccl_plan_build(C.byref(c), C.addressof(shape), nd, C.byref(plan)), "apc_nccl_plan_build")
    return plan


def upload_nccl_plan(model: _lib.ApcModel, cfg, device) -> torch.Tensor:
    """Build the plan for model's mesh, copy it to ``device`` and point
    ``model.nccl_plan`` at the copy.  The caller keeps the returned tensor alive
    for as long as the model is used."""
    plan = build_nccl_plan(cfg, [model.mesh_shape[i] for i in range(model.ndim)])
    raw = np.frombuffer(bytes(plan), dtype=np.uint8).copy()
    t = torch.from_numpy(raw).to(device)
    model.nccl_plan = t.data_ptr()
    return t


_stage = threading.local()  # .buffer: this thread's pinned staging buffer


def _upload_stage(nbytes: int) -> torch.Tensor:
    """Pinned staging buffer of the upload arena, kept between the engines a
    thread makes (pinning memory costs more than the copy it serves); an engine
    is done with it when its copy has run, before its constructor returns."""
    buf = getattr(_stage, "buffer", None)
    if buf is None or buf.numel() < nbytes:
        buf = _stage.buffer = torch.empty(max(nbytes, 1 << 20), dtype=torch.uint8, pin_memory=True)
    return buf


def detect_device_name(device=None) -> str:
    """Marketing name of the HIP device, as the reference's device table keys
    on it (autoparallel/cost_models/compute_estimation.py:258-275).  Hosts
    without the amdgpu id database report every card as "AMD Radeon Graphics";
    the architecture name then decides (gfx950 is MI355X)."""
    name = torch.cuda.get_device_name(device)
    if "Instinct" not in name:
        arch = getattr(torch.cuda.get_device_properties(device), "gcnArchName", "")
        if arch.startswith("gfx950"):
            return "AMD Instinct MI355X"
        if arch.startswith("gfx942"):
            return "AMD Instinct MI300X"
    return name


def _edit_count(t: Optional[torch.Tensor]) -> int:
    """How often torch has edited ``t`` in place; -1 where that is not counted."""
    return -1 if t is None or t.is_inference() else t._version


class CostEngine:
    def __init__(
        self,
        g: PackedGraph,
        device: str = "cuda",
        device_name: Optional[str] = None,
        use_table: Optional[bool] = None,
        order_mode: int = 0,
        nccl_config=None,
        table_mode: Optional[str] = None,
        item_entries: Optional[int] = None,
        topo_config=None,
        allocate_results: bool = True,
        lut: Optional[bool] = None,
    ):
        """``table_mode``: "full" (one S_dst x S_src matrix per distinct pair of
        runs), "compressed" (matrices by distinct spec word, read by gather),
        "direct" (no table: every entry evaluated), or None: the first of the
        three whose table is small against the entry count.  ``topo_config``:
        an XGMITopoConfig for the alpha-beta constants (make_model).
        ``allocate_results=False``: only the problem is uploaded (for the node
        hashes, which are taken before it is decided which edges get entries);
        such an engine cannot build.  ``lut``: build the block table (or, without
        one, the entries) with the lookup-table kernels; None: for tables of
        more than 2 048 units and for direct evaluation.  ``use_table`` is
        the older switch: True = "full", False = "direct".  ``item_entries``:
        entries per work item of the entry kernel, 256 or 512 (512 needs a
        table); None: by problem size."""
        self.lib = _lib.load()
        self.g = g
        self.device = torch.device(device)
        if self.device.type != "cuda":
            raise _lib.ApcError("CostEngine needs a HIP device; there is no CPU path")
        if device_name is None:
            device_name = detect_device_name(self.device)
        self.device_name = device_name
        g.validate()
        sizes = g.edge_sdst.astype(np.int64) * g.edge_ssrc
        assert g.num_edges == 0 or int(sizes.max()) < 2**31, "edge block too large for 32-bit local index"

        self._keep: Dict[str, torch.Tensor] = {}
        self._layouts: Dict[str, dict] = {"score_tiles": {}, "score_tiles_explicit": {}, "sample_steps": {},
                                          "score_pieces": {}, "piece_counts": {}, "large_block_costs": {},
                                          "sample_tiles": {}, "pair_tiles": {}}

        # The problem is some thirty arrays, most of them a few kilobytes: they go up in
        # one copy.  An array is laid into a pinned staging buffer and gets its address
        # inside a device arena at once (the struct fields below need it); the arena is
        # filled by _flush_uploads when all of them are known.  Large arrays (and what
        # does not fit any more) are copied on their own.
        arena_bytes = int(min(_UPLOAD_ARENA_BYTES, (256 << 10) + 32 * g.lists.shape[0] + 160 * g.num_edges
                              + 320 * g.num_nodes + 8 * g.default_vals.shape[0]))
        stage = _upload_stage(arena_bytes)
        arena = torch.empty(arena_bytes, dtype=torch.uint8, device=self.device)
        stage_np = stage.numpy()
        used = [0]

        def up(name, arr, dtype=None):
            a = np.ascontiguousarray(arr if dtype is None else arr.astype(dtype))
            if a.dtype == np.uint32:
                a = a.view(np.int32)
            raw = a.reshape(-1).view(np.uint8) if a.dtype.fields is None else a.view(np.uint8).reshape(-1)
            n = raw.shape[0]
            off = (used[0] + 255) & ~255
            if n == 0 or n > _UPLOAD_ARENA_MAX_ARRAY or off + n > arena_bytes:
                t = torch.from_numpy(raw if a.dtype.fields is not None else a).to(self.device)
            else:
                stage_np[off:off + n] = raw
                used[0] = off + n
                t = arena[off:off + n]
                if a.dtype.fields is None:
                    t = t.view(torch.from_numpy(a[:0].reshape(-1)).dtype).view(a.shape)
            self._keep[name] = t
            return t.data_ptr() if t.numel() else None

        def flush_uploads():
            if used[0]:
                arena[:used[0]].copy_(stage[:used[0]], non_blocking=True)
                # the staging buffer is let go once the copy has run
                torch.cuda.current_stream(self.device).synchronize()
            self._keep["upload_arena"] = arena

        p = _lib.ApcProblem()
        model = make_model([int(x) for x in g.mesh_shape], g.devices_per_host, device_name, order_mode,
                           topo_config=topo_config)
        if nccl_config is not None:  # NCCL-tuning collectives instead of alpha-beta
            self._keep["nccl_plan"] = upload_nccl_plan(model, nccl_config, self.device)
        p.model = model
        p.n_meta = g.meta_rank.shape[0]
        p.meta_rank = up("meta_rank", g.meta_rank)
        p.meta_shape = up("meta_shape", g.meta_shape)
        p.meta_stride = up("meta_stride", g.meta_stride)
        p.meta_itemsize = up("meta_itemsize", g.meta_itemsize)
        p.meta_dtype = up("meta_dtype", g.meta_dtype)
        p.n_tuple = g.tuple_plc.shape[0]
        p.tuple_plc = up("tuple_plc", g.tuple_plc)
        p.n_list = g.lists.shape[0]
        p.lists = up("lists", g.lists)
        p.n_node = g.num_nodes
        p.node_nstrat = up("node_nstrat", g.node_nstrat)
        p.node_nargs = up("node_nargs", g.node_nargs)
        p.node_op = up("node_op", g.node_op)
        p.node_comp_off = up("node_comp_off", g.node_comp_off)
        p.node_edge_off = up("node_edge_off", g.node_edge_off)
        p.node_prog_off = up("node_prog_off", g.node_prog_off)
        p.node_prog_len = up("node_prog_len", g.node_prog_len)
        p.max_node_args = g.max_node_args
        p.max_rank = g.max_rank
        p.n_compute = g.num_compute
        p.n_comp_node = g.comp_nodes.shape[0]
        p.comp_nodes = up("comp_nodes", g.comp_nodes)
        p.comp_recs = up("comp_recs", g.comp_records())
        terms, _ = g.program_terms()
        p.n_prog_term = terms.shape[0]
        p.prog_terms = up("prog_terms", terms)
        p.spec_recs = up("spec_recs", g.spec_records())
        p.max_nstrat = int(g.node_nstrat[g.comp_nodes].max()) if g.comp_nodes.shape[0] else 1
        mult = g.node_multiplier if g.node_multiplier is not None else np.ones(g.num_nodes, np.int32)
        p.node_multiplier = up("node_multiplier", mult)
        p.n_prog = g.prog.shape[0]
        p.prog = up("prog", g.prog)
        p.explicit_flops = up("explicit_flops", g.explicit_flops) if g.explicit_flops is not None else None
        p.explicit_bytes = up("explicit_bytes", g.explicit_bytes) if g.explicit_bytes is not None else None
        p.n_edge = g.num_edges
        p.n_entry = g.num_entries
        p.n_slot = g.num_slots
        chunk_edge = g.chunk_edge_index()
        p.n_chunk = chunk_edge.shape[0]
        assert p.n_chunk == g.num_slots >> CHUNK_SHIFT
        p.chunk_edge = up("chunk_edge", chunk_edge)
        signed_defaults = bool(np.signbit(g.default_vals).any())
        if table_mode is None and use_table is not None:
            table_mode = "full" if use_table else "direct"
        if table_mode is None:
            table_mode = g.default_table_mode()
        if table_mode not in ("direct", "full", "compressed"):
            raise ValueError(f"unknown table_mode {table_mode!r}")
        if table_mode != "direct" and signed_defaults:
            raise ValueError("a block table needs default values with a clear sign bit")
        self.table_mode = table_mode
        squeezed = table_mode == "compressed"
        p.edges = up("edges", g.edge_records(squeezed))
        self.item_entries = g.default_item_entries(table_mode) if item_entries is None else int(item_entries)
        items = g.work_items(squeezed, self.item_entries)
        p.item_entries = self.item_entries
        p.n_item = items.shape[0]
        p.items = up("items", items)
        p.n_default = g.default_vals.shape[0]
        p.default_vals = up("default_vals", g.default_vals)
        block_edge, block_off, unit_block, _, _, block_udst = g.block_table(squeezed)
        if squeezed:
            uidx, ufirst, _ = g.run_unique_index()
            p.list_uidx = up("list_uidx", uidx)
            p.list_ufirst = up("list_ufirst", ufirst)
            p.block_udst = up("block_udst", block_udst)
        p.n_block = block_edge.shape[0]
        p.block_edge = up("block_edge", block_edge)
        p.block_off = up("block_off", block_off)
        p.table_size = int(block_off[-1])
        p.n_table_unit = unit_block.shape[0]
        p.table_unit_block = up("table_unit_block", unit_block)
        p.table_units = up("table_units", g.table_unit_records(squeezed))
        self.problem = p
        # Large tables, and direct evaluation, go through the lookup-table kernels:
        # tiles of whole matrices instead of one element per lane.
        # The library takes that route by itself when the problem carries the tile list.
        self._lut_tiles = None
        self.lut = lut if lut is not None else (table_mode == "direct" or p.n_table_unit > _LUT_TABLE_FROM)
        if self.lut and g.num_entries > 0:
            tiles = g.lut_tiles(squeezed, entries=(table_mode == "direct"))
            self._lut_tiles = (up("lut_tiles", tiles), int(tiles.shape[0]))
            if table_mode == "direct":
                p.lut_entry_tiles, p.n_lut_entry_tile = self._lut_tiles
            else:
                p.lut_table_tiles, p.n_lut_table_tile = self._lut_tiles
        flush_uploads()

        E, NC = (g.num_slots, g.num_compute) if allocate_results else (0, 0)
        self.can_build = bool(allocate_results)
        # entry arrays hold num_slots elements; padding slots stay zero
        self.compute = torch.zeros(NC, dtype=torch.float64, device=self.device)
        self.per_arg = torch.zeros(NC, dtype=torch.float64, device=self.device)
        self.comm = torch.zeros(E, dtype=torch.float64, device=self.device)
        self.cost = torch.zeros(E, dtype=torch.float64, device=self.device)
        self.flags = torch.zeros(E, dtype=torch.uint8, device=self.device)
        self.status = torch.zeros(1, dtype=torch.int32, device=self.device)
        tsize = int(self.lib.apc_pair_table_size(C.byref(p)))
        self.use_table = table_mode != "direct"
        self.table = (
            torch.empty(tsize, dtype=torch.float64, device=self.device)
            if self.use_table and allocate_results else None
        )
        self.built = False
        self._build_args = None
        # Batches of _SCORE_LANES_FROM assignments and more are scored from something
        # denser than the three entry arrays: the block table itself when the blocks
        # are large (_score_packed), else records made from the arrays on first use,
        # stale after anything rewrites the arrays.
        self.packed_scoring = g.num_edges > 0 and g.num_entries > 0
        self._whole_walk = self._walk_from(0)
        self.large_blocks = g.num_edges > 0 and g.num_entries / g.num_edges >= _LARGE_BLOCKS_FROM
        self._recs: Optional[torch.Tensor] = None
        self._recs_valid = False
        self._recs_compact = False
        # clamp_inf of the build whose table path wrote the entry arrays as they are now,
        # None once anything else has written them: then scoring cannot read the table instead
        self._table_clamp: Optional[int] = None
        # and the arrays builds write, with their version counters: another tensor put in the place of
        # one, or a caller's edit in place, shows by them (tensors made under inference_mode have no
        # counters); the same of the arrays that the records were made from.  A build takes the counters
        # again only for a caller who has been seen to edit (a build of a small graph is bound by its
        # host time, of which the four counters are 2%): after a first edit that only a build, and no
        # scoring, has followed, scoring reads the arrays until the next build.
        self._versioned = not self.comm.is_inference()
        self._edits_seen = False
        # what launches that write the arrays and were recorded in a graph leave in them whenever it is
        # replayed: the clamp_inf of a build, None for anything else
        self._recorded_writes: set = set()
        self._built_marks = self._array_marks()
        self._recs_marks: tuple = ()
        self.last_score_backend = "entry_arrays"  # what the last batch was scored from
        self.last_score_entry = ""  # and by which entry point of the library
        self.last_sample_backend = ""  # how the last feasible draws were made: by "tiles", "steps" or "lanes"

    def synchronize(self) -> None:
        torch.cuda.synchronize(self.device)

    # -- raw stream -----------------------------------------------------------
    # The handle alone: a torch.cuda.Stream made for every call costs 3 us of host time, a third
    # of what issuing a build takes.
    def _raw_stream(self) -> int:
        index = self.device.index
        return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if index is None else index)

    def _stream(self):
        return C.c_void_p(self._raw_stream())

    @staticmethod
    def _ptr(t: Optional[torch.Tensor]):
        return None if t is None or t.numel() == 0 else C.c_void_p(t.data_ptr())

    # -- kernels --------------------------------------------------------------
    def build_pair_table(self):
        if self.table is not None:
            _lib.check(
                self.lib.apc_build_pair_table(C.byref(self.problem), self._ptr(self.table), self._stream()),
                "apc_build_pair_table",
            )

    def node_compute(self):
        _lib.check(
            self.lib.apc_node_compute_costs(
                C.byref(self.problem), self._ptr(self.compute), self._ptr(self.per_arg),
                self._ptr(self.status), self._stream()),
            "apc_node_compute_costs",
        )

    def _capturing(self, stream) -> bool:
        """Whether ``stream``, the current one (_stream()), records its launches in a graph."""
        if not stream.value:  # the default stream never does
            return False
        with torch.cuda.device(self.device):
            return torch.cuda.is_current_stream_capturing()

    def _arrays_rewritten(self, stream) -> None:
        """Something else than a build writes the arrays: now, or whenever a graph is replayed."""
        self._recs_valid = False
        self._table_clamp = None
        if self._capturing(stream):
            self._recorded_writes.add(None)

    def mark_results_edited(self) -> None:
        """To be called by a caller that has written into comm / cost / flags / per_arg
        itself: scoring then reads the arrays as they are (records are made again on the
        next large batch, and the block table no longer stands for the arrays).  Edits that
        a graph makes when it is replayed are marked after the replay, or once for all
        while they are recorded."""
        self._edits_seen = True
        self._arrays_rewritten(self._stream())

    def edge_costs(self, clamp_inf: bool = True, want_comm: bool = True, want_flags: bool = True):
        stream = self._stream()
        self._arrays_rewritten(stream)
        _lib.check(
            self.lib.apc_edge_costs(
                C.byref(self.problem), self._ptr(self.table), self._ptr(self.per_arg),
                self._ptr(self.comm) if want_comm else None, self._ptr(self.cost),
                self._ptr(self.flags) if want_flags else None, int(bool(clamp_inf)), stream),
            "apc_edge_costs",
        )

    def edge_costs_timed(self, timer, slot: int, clamp_inf: bool = True):
        """edge_costs with HIP events at the kernel's begin and end (a timer from
        apc_timer_create); the launch is otherwise identical."""
        stream = self._stream()
        self._arrays_rewritten(stream)
        _lib.check(
            self.lib.apc_edge_costs_timed(
                C.byref(self.problem), self._ptr(self.table), self._ptr(self.per_arg), self._ptr(self.comm),
                self._ptr(self.cost), self._ptr(self.flags), int(bool(clamp_inf)), timer, int(slot), stream),
            "apc_edge_costs_timed",
        )

    def prepare(self):
        """Pair table and node compute vectors, as build() makes them: one launch,
        or, with the lookup-table kernels, the table by tiles and the node launch."""
        _lib.check(
            self.lib.apc_prepare(
                C.byref(self.problem), self._ptr(self.table), self._ptr(self.compute),
                self._ptr(self.per_arg), self._ptr(self.status), self._stream()),
            "apc_prepare",
        )

    def build_args(self):
        if not self.can_build:
            raise _lib.ApcError("this engine holds the problem only (allocate_results=False)")
        if self._build_args is None:
            self._build_args = (
                C.byref(self.problem), self._ptr(self.table), self._ptr(self.compute), self._ptr(self.per_arg),
                self._ptr(self.status), self._ptr(self.comm), self._ptr(self.cost), self._ptr(self.flags))
        return self._build_args

    def build(self, clamp_inf: bool = True):
        """All coefficients: pair table and node compute vectors, then the entry
        arrays (apc_build_all: two launches, three when the table is built by tiles)."""
        self._recs_valid = False
        # the argument list is the same from call to call apart from the stream:
        # made once, so that issuing a step costs less host time than the step takes
        args = self._build_args or self.build_args()
        stream = self._raw_stream()
        rc = self.lib.apc_build_all(*args, 1 if clamp_inf else 0, stream)
        if rc:
            _lib.check(rc, "apc_build_all")
        self.built = True
        self._note_build((1 if clamp_inf else 0) if self.table is not None else None, stream)
        return self

    def build_timed(self, timer, slot: int, clamp_inf: bool = True):
        """build() with HIP events at the begin and end of the kernel that writes
        the entries (a timer from apc_timer_create); the launches are otherwise
        identical."""
        self.build_args()
        stream = self._raw_stream()
        clamp = 1 if clamp_inf else 0
        rc = self.lib.apc_build_all_timed(*self._build_args, clamp, timer, int(slot), stream)
        if rc:
            _lib.check(rc, "apc_build_all_timed")
        self._recs_valid = False
        self.built = True
        self._note_build(clamp if self.table is not None else None, stream)
        return self

    def _note_build(self, clamp: Optional[int], stream: int) -> None:
        if stream and self._capturing(C.c_void_p(stream)):  # nothing is written yet
            self._recorded_writes.add(clamp)
            return
        self._table_clamp = clamp
        if self._edits_seen:  # edits before this build are gone
            self._built_marks = tuple((ref, at, _edit_count(ref())) for ref, at, _ in self._built_marks)

    def set_node_multiplier(self, mult: np.ndarray) -> None:
        """Replace the objective multiplier per node (cluster multiplicity)."""
        t = self._keep["node_multiplier"]
        assert len(mult) == t.numel()
        t.copy_(torch.from_numpy(np.ascontiguousarray(mult, np.int32)))

    def load_results(self, comm, cost, flags, compute, per_arg):
        """Adopt coefficient arrays computed earlier (a saved optimizer): host
        arrays of num_slots / num_compute elements are copied to the device and
        the engine counts as built.  Nothing is recomputed."""
        g = self.g
        assert len(comm) == len(cost) == len(flags) == g.num_slots and len(compute) == len(per_arg) == g.num_compute
        self.comm.copy_(torch.from_numpy(np.ascontiguousarray(comm, np.float64)))
        self.cost.copy_(torch.from_numpy(np.ascontiguousarray(cost, np.float64)))
        self.flags.copy_(torch.from_numpy(np.ascontiguousarray(flags, np.uint8)))
        self.compute.copy_(torch.from_numpy(np.ascontiguousarray(compute, np.float64)))
        self.per_arg.copy_(torch.from_numpy(np.ascontiguousarray(per_arg, np.float64)))
        self.built = self._edits_seen = True
        self._arrays_rewritten(self._stream())
        return self

    def capture_build(self, clamp_inf: bool = True) -> "torch.cuda.CUDAGraph":
        """The launches of build() recorded in a HIP graph, for callers that
        replay a whole planning step from a graph.  On its own a replay is no
        faster than the eager launches (measured on the headline graph: 29.8 us
        a replay against 25.8 us for the two launches issued eagerly with cached
        argument lists).  The graph holds kernel nodes only (no memset nodes);
        it is valid while this engine's buffers live.  build() is run once
        eagerly first so that one-time function attributes are set outside the
        capture.  Scoring takes into account that a replay may have followed the
        last eager build."""
        self.build(clamp_inf)
        torch.cuda.synchronize(self.device)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            self.build(clamp_inf)
        return graph

    def check_status(self):
        if int(self.status.item()) != 0:
            raise ValueError(
                "a node with flops has an input dtype without a tflops entry on "
                f"{self.device_name} (the reference raises ValueError for it)"
            )

    def apply_prefetch_discount(self, scale: float = 0.0) -> int:
        assert self.built
        stream = self._stream()
        self._arrays_rewritten(stream)
        n = torch.zeros(1, dtype=torch.int64, device=self.device)
        _lib.check(
            self.lib.apc_apply_prefetch_discount(
                C.byref(self.problem), self._ptr(self.per_arg), float(scale), self._ptr(self.comm),
                self._ptr(self.cost), self._ptr(self.flags), self._ptr(n), stream),
            "apc_apply_prefetch_discount",
        )
        return int(n.item())

    def objective_coeffs(self) -> torch.Tensor:
        assert self.built
        obj = torch.empty_like(self.cost)  # the pass writes every slot, zero between the blocks
        if self.g.num_entries == 0:
            return obj.zero_()
        _lib.check(
            self.lib.apc_objective_coeffs(C.byref(self.problem), self._ptr(self.cost), self._ptr(obj), self._stream()),
            "apc_objective_coeffs",
        )
        return obj

    def score(self, assign: torch.Tensor) -> torch.Tensor:
        """assign: uint16/int16 [n_node, n_assign] on the device -> float64 [n_assign, 6]."""
        assert self.built
        assert assign.dim() == 2 and assign.shape[0] == self.g.num_nodes and assign.is_contiguous()
        assert assign.dtype in (torch.int16, torch.uint16) and assign.device == self.comm.device
        A = assign.shape[1]
        out = torch.empty((A, 6), dtype=torch.float64, device=self.device)
        if self.packed_scoring and A >= _SCORE_LANES_FROM:
            return self._score_packed(assign, 0, 0, A, None, 0, None, out)
        return self._score_small(assign, 0, 0, A, None, 0, None, out)

    def _array_marks(self) -> tuple:
        return tuple((weakref.ref(t), t.data_ptr(), _edit_count(t))
                     for t in (self.comm, self.cost, self.flags, self.per_arg))

    def _unchanged(self, marks: tuple) -> bool:
        """Whether the arrays are the marked ones, with no edit since."""
        arrays = (self.comm, self.cost, self.flags, self.per_arg)
        for (ref, at, n), t in zip(marks, arrays):
            if ref() is not t or t.data_ptr() != at or (n >= 0 and t._version != n):
                return False
        return len(marks) > 0

    def _standing_clamp(self) -> Optional[int]:
        """clamp_inf of the build that made the entry arrays what they are, while they still are what
        it made of the block table, so that a scorer may read the table in their place; else
        None.  Every scorer that does so asks here.  Recorded builds may have been replayed since the
        last one: they change nothing where they clamp alike."""
        if self._table_clamp is None or self._recorded_writes - {self._table_clamp}:
            return None
        if self._unchanged(self._built_marks):
            return self._table_clamp
        self._edits_seen = True
        return None

    def _score_small(self, assign, seed, first, count, d_gid, first_node, init, out) -> torch.Tensor:
        """A batch below _SCORE_LANES_FROM: the terms side by side, from the block table while it stands for
        the entry arrays, else from the arrays."""
        stream = self._stream()
        if _SCORE_SMALL_FROM_TABLE and self.packed_scoring and count > 0:
            # recorded, it reads whatever the arrays hold on a replay; without edit counters, an edit
            # would go unnoticed
            clamp = self._standing_clamp() if self._versioned and not self._capturing(stream) else None
            if clamp is not None:
                return self._score_terms(clamp, assign, seed, first, count, d_gid, first_node, init, out, stream)
        return self._score_arrays(assign, seed, first, count, d_gid, first_node, init, out, stream)

    def _launch_score(self, name: str, *args) -> None:
        _lib.check(getattr(self.lib, name)(*args), name)
        self.last_score_entry = name

    def _score_arrays(self, assign, seed, first, count, d_gid, first_node, init, out, stream) -> torch.Tensor:
        args = (C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self.comm), self._ptr(self.cost),
                self._ptr(self.flags))
        if assign is not None:
            self.last_score_entry = "apc_score_assignments_window"
            rc = self.lib.apc_score_assignments_window(
                *args, self._ptr(assign), int(count), int(first_node), self._ptr(init), self._ptr(out), stream)
        elif d_gid is None:
            self.last_score_entry = "apc_score_random_assignments"
            rc = self.lib.apc_score_random_assignments(*args, int(seed), int(first), int(count), self._ptr(out), stream)
        else:
            self.last_score_entry = "apc_score_random_window"
            rc = self.lib.apc_score_random_window(
                *args, int(seed), int(first), int(count), self._ptr(d_gid), int(first_node), self._ptr(init),
                self._ptr(out), stream)
        _lib.check(rc, self.last_score_entry)
        self.last_score_backend = "entry_arrays"
        return out

    def _walk_from(self, first_node: int):
        """(first edge, edges, nodes) of the walk from ``first_node`` on."""
        first_edge = int(self.g.node_edge_off[first_node])
        return first_edge, self.g.num_edges - first_edge, self.g.num_nodes - first_node

    def _score_terms(self, clamp, assign, seed, first, count, d_gid, first_node, init, out, stream) -> torch.Tensor:
        g = self.g
        first_edge, n_edge, n_node = self._whole_walk if first_node == 0 else self._walk_from(first_node)
        few, scratch = 0, None
        for most, small, large in _SCORE_TERM_FIELDS_UP_TO:
            if count <= most:
                few = large if self.large_blocks else small
                break
        if _SCORE_TERM_RECORDS and n_edge > 0 and n_node > 0 and (n_edge > few or n_node > few):
            scratch = self._scratch(n_edge * _lib.FOLD_EDGE_BYTES + n_node * _lib.FOLD_NODE_BYTES)
        if scratch is not None:
            self.last_score_entry = "apc_score_terms"
            rc = self.lib.apc_score_terms(
                C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self.table), self._ptr(scratch),
                self._ptr(assign), int(seed), int(first), int(count), self._ptr(d_gid), int(first_node), first_edge,
                clamp, self._ptr(init), self._ptr(out), stream)
        else:
            self.last_score_entry = "apc_score_fold_table"
            rc = self.lib.apc_score_fold_table(
                C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self.table), self._ptr(assign), int(seed),
                int(first), int(count), self._ptr(d_gid), int(first_node), clamp, self._ptr(init),
                self._ptr(out), stream)
        _lib.check(rc, self.last_score_entry)
        self.last_score_backend = "block_table_terms"
        return out

    def _score_packed(self, assign, seed, first, count, d_gid, first_node, init, out) -> torch.Tensor:
        """Scoring of a large batch.  A graph with large blocks: from the block
        table while the entry arrays are what the last build made of it
        (apc_score_stream, or apc_score_table for explicit assignments, more strategies than that takes, and where
        large_block_costs says so; 5x the rate of any walk over records there).  Else,
        and for graphs with small blocks: up to _SCORE_TERMS_UP_TO_IMAGES assignments with
        the terms gathered side by side from the table (apc_score_terms), from
        there on by tiles of edges (random ones apc_score_pairs: 7.2 ms for 2^20 assignments of the Llama-3-8B graph,
        against 10.4 by apc_score_from_tiles, which takes random ones that carry sums, 15.6 ms from records, 18.0 ms from
        the table edge by edge and 31.2 ms from the three arrays; explicit ones, and up to _SCORE_IMAGES_UP_TO that carry
        sums, apc_score_images).  Where the table does not
        stand for the arrays, or the graph has no such tiles: from records made here if the entry
        arrays changed since: compact 16-byte
        records, several assignments per lane (apc_score_compact), while every
        cost is (comm + per_arg) + transition or its clamp (checked on the device
        when the records are made); else the 32-byte records that carry the cost
        (apc_score_packed)."""
        g = self.g
        stream = self._stream()
        capturing = self._capturing(stream)
        clamp = self._standing_clamp() if _SCORE_FROM_TABLE else None
        from_table = clamp is not None
        large = self.large_blocks or not _SCORE_COMPACT
        pieces = None
        table_from = _SCORE_TABLE_FROM
        if from_table and large and count >= table_from and self._versioned:
            if assign is not None:
                table_from *= _SCORE_TABLE_EXPLICIT
            else:
                counts = None
                if _SCORE_STREAM:
                    counts = self._layout("piece_counts", first_node, lambda: piece_counts(g, self._matrix_sizes(), first_node))
                edge_by_edge_us = self._edge_by_edge_us(counts, first_node, count, capturing)
                if edge_by_edge_us is not None:
                    table_from = max(table_from, 1e6 * edge_by_edge_us[0] / edge_by_edge_us[1])
                elif counts is not None:
                    table_from *= max(1.0, counts[0] / counts[1] / _SCORE_TABLE_PIECES)
                    if count >= table_from:  # else the list need not be made
                        pieces = self._score_pieces(first_node)
                if pieces is None and edge_by_edge_us is None:
                    table_from = max(table_from, _SCORE_TABLE_FROM * _SCORE_TABLE_EDGES)
        if from_table and large and count >= table_from:
            if pieces is not None:
                d_pieces, n_piece, n_item = pieces
                scratch = self._scratch(n_item * _lib.SCORE_SIDE_BYTES + n_piece * _lib.SCORE_PIECE_SCRATCH)
                if scratch is not None:
                    self._launch_score(
                        "apc_score_stream",
                        C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self.table), self._ptr(d_pieces),
                        n_piece, n_item, self._ptr(scratch), int(seed), int(first), int(count), self._ptr(d_gid),
                        clamp, self._ptr(init), self._ptr(out), stream)
                    self.last_score_backend = "block_table"
                    return out
            aux = self._score_edge_aux(d_gid)
            self._launch_score(
                "apc_score_table",
                C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self.table),
                C.c_void_p(aux.data_ptr()), self._ptr(assign),
                int(seed), int(first), int(count), self._ptr(d_gid), int(first_node), self.g.num_nodes,
                clamp, min(_SCORE_PER_LANE, 4),
                self._ptr(init), self._ptr(out), stream)
            self.last_score_backend = "block_table"
            return out
        from_table &= self._versioned  # else an edit would go unnoticed
        if from_table and _SCORE_FROM_TILES and not self.large_blocks and _SCORE_PAIRS and (
                assign is None and init is None and count > _SCORE_PAIRS_FROM[
                    0 if g.num_entries * _SCORE_PAIRS_ROWS <= g.num_edges * _lib.PAIR_TILE_UNITS else 1]):
            pairs = self._pair_tiles(first_node)
            if pairs is not None and pairs[3] >= _SCORE_PAIRS_TILES:
                steps, n_step, d_tiles, n_tile = pairs
                scratch = self._scratch((n_tile + 1) * _lib.PAIR_IMAGE_BYTES)
                if scratch is not None:
                    self._launch_score(
                        "apc_score_pairs",
                        C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self.table), self._ptr(steps),
                        n_step, self._ptr(d_tiles), n_tile, self._ptr(scratch), int(seed), int(first), int(count),
                        self._ptr(d_gid), clamp, self._ptr(out), stream)
                    self.last_score_backend = "block_table_tiles"
                    return out
        terms_up_to, kind = -1, "random" if assign is None else "explicit"
        if _SCORE_SMALL_FROM_TABLE and _SCORE_TERMS_ABOVE:
            terms_up_to = _SCORE_TERMS_UP_TO_IMAGES[kind]
        by_tiles = from_table and _SCORE_FROM_TILES and not self.large_blocks and count > terms_up_to
        if by_tiles and assign is not None and terms_up_to >= 0 and count <= _SCORE_TERMS_UP_TO_IMAGES["random"]:
            tiles = self._score_tiles(first_node, True)
            by_tiles = tiles is None or self._walk_from(first_node)[1] >= tiles[3] * _SCORE_IMAGES_EDGES
        if by_tiles:
            name, scratch = "apc_score_images", None
            if assign is not None or count <= _SCORE_IMAGES_UP_TO:
                tiles = self._score_tiles(first_node, True)
                if tiles is not None and (tiles[3] >= _SCORE_IMAGES_TILES or count <= 1 << 18):
                    scratch = self._scratch((tiles[3] + 1) * _lib.SCORE_IMAGE_BYTES)
            if scratch is None:
                name, tiles = "apc_score_from_tiles", self._score_tiles(first_node, assign is not None)
                if tiles is not None:
                    scratch = self._scratch(tiles[1] * _lib.SCORE_STEP_BYTES)
            if scratch is not None:
                steps, n_step, d_tiles, n_tile, units = tiles
                self._launch_score(
                    name,
                    C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self.table), self._ptr(steps), n_step,
                    self._ptr(d_tiles), n_tile, self._ptr(units), self._ptr(scratch), self._ptr(assign),
                    int(seed), int(first), int(count), self._ptr(d_gid), clamp, self._ptr(init),
                    self._ptr(out), stream)
                self.last_score_backend = "block_table_tiles"
                return out
        # on a graph with large blocks, what is not scored by the table above
        if from_table and terms_up_to >= 0 and (large or count <= _SCORE_TERMS_UP_TO_RECORDS[kind]):
            return self._score_terms(clamp, assign, seed, first, count, d_gid, first_node, init, out, stream)
        recs_stand = (self._recs_valid and self._unchanged(self._recs_marks)
                      and (capturing or not self._recorded_writes))  # else replayed since, or not
        if capturing and not recs_stand:  # records are not made meanwhile: the host reads their check
            return self._score_arrays(assign, seed, first, count, d_gid, first_node, init, out, stream)
        if not recs_stand:
            self._recs = None  # one kind at a time: either is as large as the entry arrays
            recs = None
            self._recs_compact = False
            if _SCORE_COMPACT:
                recs = torch.empty(self.g.num_slots * 2, dtype=torch.float64, device=self.device)
                mismatch = torch.empty(1, dtype=torch.int32, device=self.device)
                _lib.check(
                    self.lib.apc_pack_score_records16(
                        C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self.comm), self._ptr(self.cost),
                        self._ptr(self.flags), self._ptr(recs), self._ptr(mismatch), self._stream()),
                    "apc_pack_score_records16")
                self._recs_compact = int(mismatch.item()) == 0
            if not self._recs_compact:
                del recs
                recs = torch.empty(self.g.num_slots * 4, dtype=torch.float64, device=self.device)
                _lib.check(
                    self.lib.apc_pack_score_records(
                        C.byref(self.problem), self._ptr(self.comm), self._ptr(self.cost), self._ptr(self.flags),
                        self._ptr(recs), self._stream()),
                    "apc_pack_score_records")
            self._recs = recs
            self._recs_valid = True
            self._recs_marks = self._array_marks()
        if self._recs_compact:
            self._launch_score(
                "apc_score_compact",
                C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self._recs), self._ptr(assign),
                int(seed), int(first), int(count), self._ptr(d_gid), int(first_node), self.g.num_nodes,
                _SCORE_PER_LANE, self._ptr(init), self._ptr(out), self._stream())
            self.last_score_backend = "compact_records"
            return out
        self._launch_score(
            "apc_score_packed",
            C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self._recs), self._ptr(assign),
            int(seed), int(first), int(count), self._ptr(d_gid), int(first_node), self._ptr(init),
            self._ptr(out), self._stream())
        self.last_score_backend = "records"
        return out

    def _scratch(self, nbytes: int) -> Optional[torch.Tensor]:
        """Scratch of a call, or None where the device has no room for it: the caller then takes a way that needs
        less."""
        try:
            return torch.empty(nbytes, dtype=torch.uint8, device=self.device)
        except torch.cuda.OutOfMemoryError:
            return None

    def _score_tiles(self, first_node: int, explicit: bool):
        """The layout apc_score_from_tiles walks from ``first_node`` on (apc_score_images: one made with
        ``explicit``), on the device, or None:
        a graph that form does not take, or no layout at hand (_layout)."""
        return self._layout("score_tiles_explicit" if explicit else "score_tiles", first_node,
                            lambda: self._make_score_tiles(first_node, explicit))

    def _layout(self, kind: str, first_node: int, make):
        """``make()`` for the walk from ``first_node`` on, made once.  None too once
        _LAYOUTS_KEPT have been made, and while a graph is recorded, where nothing can be copied to
        the device."""
        kept = self._layouts[kind]
        if first_node in kept:
            return kept[first_node]
        if len(kept) >= _LAYOUTS_KEPT or self._capturing(self._stream()):
            return None
        return kept.setdefault(first_node, make())

    def _make_score_tiles(self, first_node: int, explicit: bool):
        g = self.g
        plan = None
        if self.table_mode == "full" and first_node < g.num_nodes:
            edges = np.ascontiguousarray(g.edge_records(False))
            a = [np.ascontiguousarray(x, t) for x, t in (
                (g.node_edge_off, np.int32), (g.node_nstrat, np.int32), (g.node_nargs, np.int32),
                (g.node_comp_off, np.int64))]
            max_step, max_unit = score_tile_room(g)
            steps = np.empty((max_step, _lib.SCORE_STEP_BYTES), np.uint8)
            tiles = np.empty((max_step, _lib.SCORE_TILE_BYTES), np.uint8)
            units = np.empty((max_unit, _lib.SCORE_UNIT_BYTES), np.uint8)
            n = [C.c_int32(0) for _ in range(3)]
            _lib.check(
                self.lib.apc_score_tiles(
                    edges.ctypes.data, g.num_edges, g.num_nodes, *[x.ctypes.data for x in a], int(first_node),
                    int(explicit), steps.ctypes.data, max_step, tiles.ctypes.data, max_step, units.ctypes.data,
                    max_unit, *[C.byref(x) for x in n]),
                "apc_score_tiles")
            n_step, n_tile, n_unit = [x.value for x in n]
            if n_step > 0:
                plan = (torch.from_numpy(steps[:n_step]).to(self.device), n_step,
                        torch.from_numpy(tiles[:n_tile]).to(self.device), n_tile,
                        torch.from_numpy(units[:n_unit]).to(self.device))
        return plan

    def _pair_tiles(self, first_node: int):
        """The layout apc_score_pairs walks from ``first_node`` on, on the device, or None: a graph that form does not
        take, or no layout at hand (_layout)."""
        return self._layout("pair_tiles", first_node, lambda: self._make_pair_tiles(first_node))

    def _make_pair_tiles(self, first_node: int):
        g = self.g
        if self.table_mode != "full" or first_node >= g.num_nodes:
            return None
        edges = np.ascontiguousarray(g.edge_records(False))
        off, nstrat = [np.ascontiguousarray(x, np.int32) for x in (g.node_edge_off, g.node_nstrat)]
        most = g.num_nodes + g.num_edges
        steps = np.empty((most, _lib.PAIR_STEP_BYTES), np.uint8)
        tiles = np.empty((most, _lib.PAIR_TILE_BYTES), np.uint8)
        n_step, n_tile = C.c_int32(0), C.c_int32(0)
        _lib.check(
            self.lib.apc_pair_tiles(
                edges.ctypes.data, g.num_edges, g.num_nodes, off.ctypes.data, nstrat.ctypes.data, int(first_node),
                steps.ctypes.data, most, tiles.ctypes.data, most, C.byref(n_step), C.byref(n_tile)),
            "apc_pair_tiles")
        if n_tile.value == 0:
            return None
        return (torch.from_numpy(steps[:n_step.value]).to(self.device), n_step.value,
                torch.from_numpy(tiles[:n_tile.value]).to(self.device), n_tile.value)

    def _score_pieces(self, first_node: int):
        """(apc_score_piece records on the device, pieces, items) of apc_score_stream for the walk from
        ``first_node`` on, or None: a node with too many strategies, nothing to score, or no layout at hand."""
        return self._layout("score_pieces", first_node, lambda: self._make_score_pieces(first_node))

    def _edge_by_edge_us(self, counts, first_node: int, count: int, capturing: bool):
        """(us an edge, ns the terms of one take for 1 000 assignments) where ``count`` random assignments are faster from the
        table edge by edge than as a stream of the pieces of ``counts``, else None."""
        if counts is None or (capturing and "score_edge_aux" not in self._keep):  # its records cannot be made meanwhile
            return None
        costs = self._layout("large_block_costs", first_node, lambda: large_block_costs(
            counts, self._matrix_sizes()[self.g.node_edge_off[first_node]:], int(self.lib.apc_score_table_tile()),
            self.table.numel() * 8e-6))
        if costs is None:
            return None
        (stream, stream_top), (table, table_top, table_top2), terms = costs
        filled = max(min(count, 1 << 20) - (1 << 18), 0) / ((1 << 20) - (1 << 18))
        table += (table_top + table_top2 * filled) * filled
        return (table, terms) if table < stream + stream_top * filled else None

    def _matrix_sizes(self) -> np.ndarray:
        if "matrix_sizes" not in self._keep:
            self._keep["matrix_sizes"] = matrix_sizes(self.g, self.table_mode == "compressed")
        return self._keep["matrix_sizes"]

    def _make_score_pieces(self, first_node: int):
        g = self.g
        compressed = self.table_mode == "compressed"
        size = self._matrix_sizes()
        if size.max(initial=0) > 0x7FFFFFFF - _lib.SCORE_PIECE:
            return None
        size = size.astype(np.int32)
        edges = np.ascontiguousarray(g.edge_records(compressed))
        off, nstrat = [np.ascontiguousarray(x, np.int32) for x in (g.node_edge_off, g.node_nstrat)]
        most = int((size // _lib.SCORE_PIECE + 1).sum()) + g.num_nodes
        pieces = np.empty((most, _lib.SCORE_PIECE_BYTES), np.uint8)
        n_piece, n_item = C.c_int32(0), C.c_int32(0)
        _lib.check(
            self.lib.apc_score_pieces(
                edges.ctypes.data, g.num_edges, g.num_nodes, off.ctypes.data, nstrat.ctypes.data, size.ctypes.data,
                int(first_node), pieces.ctypes.data, most, C.byref(n_piece), C.byref(n_item)),
            "apc_score_pieces")
        if n_piece.value == 0:
            return None
        return torch.from_numpy(pieces[:n_piece.value]).to(self.device), n_piece.value, n_item.value

    def _score_msize(self) -> np.ndarray:
        """int32[num_edges]: the padded size of an edge's matrix in the block table
        if it is worth taking through LDS (_SCORE_STAGE_TILES tiles at most), else 0."""
        g = self.g
        _, block_off, _, edge_table_off, _, _ = g.block_table(self.table_mode == "compressed")
        msize = np.zeros(g.num_edges, np.int32)
        has = edge_table_off >= 0
        b = np.searchsorted(block_off, edge_table_off[has], side="right") - 1
        size = (block_off[b + 1] - block_off[b]).astype(np.int64)
        limit = _SCORE_STAGE_TILES * int(self.lib.apc_score_table_tile())
        msize[has] = np.where(size <= limit, size, 0).astype(np.int32)
        return msize

    def _score_edge_aux(self, d_gid: Optional[torch.Tensor]) -> torch.Tensor:
        """apc_score_edge_aux records of apc_score_table (int32[num_edges + 1, 4] on
        the device): what does not depend on the call is made once; the producers'
        ids for the draw follow the call's node ids."""
        g = self.g
        base = self._keep.get("score_edge_aux")
        if base is None:
            msize = self._score_msize()
            idx = np.where(msize > 0, np.arange(g.num_edges), g.num_edges)
            nxt = np.minimum.accumulate(np.concatenate([idx, [g.num_edges]])[::-1])[::-1]
            aux = np.zeros((g.num_edges + 1, 4), np.int32)
            aux[:-1, 0] = msize
            aux[:, 1] = np.where(nxt < g.num_edges, nxt, -1)
            aux[:-1, 2] = g.edge_src_node
            base = self._keep["score_edge_aux"] = torch.from_numpy(aux).to(self.device)
            self._keep["score_edge_src"] = torch.from_numpy(
                np.maximum(g.edge_src_node, 0).astype(np.int64)).to(self.device)
        if d_gid is None:
            return base
        aux = base.clone()
        aux[:-1, 2] = d_gid[self._keep["score_edge_src"]]
        return aux

    def node_hashes(self, node_phase: Optional[np.ndarray] = None) -> np.ndarray:
        """uint64[n_node] structural hash of every node (the clustering key).
        Needs only the uploaded problem, not the coefficients."""
        g = self.g
        out_list = torch.from_numpy(np.ascontiguousarray(g.node_out_list, np.int64)).to(self.device)
        phase = None
        if node_phase is not None:
            phase = torch.from_numpy(np.ascontiguousarray(node_phase, np.int32)).to(self.device)
        out = torch.empty(g.num_nodes, dtype=torch.int64, device=self.device)
        _lib.check(
            self.lib.apc_node_hashes(C.byref(self.problem), self._ptr(out_list), self._ptr(phase), self._ptr(out),
                                     self._stream()),
            "apc_node_hashes",
        )
        return out.cpu().numpy().view(np.uint64)

    def export_decision_vars(self):
        """(keys int32[E, 4], vals float64[E, 3]) on the device: the packed twin
        of the reference's ``decision_vars`` in its insertion order."""
        assert self.built
        if "export_row_base" not in self._keep:
            base, stride = self.g.export_rows()
            self._keep["export_row_base"] = torch.from_numpy(base).to(self.device)
            self._keep["export_row_stride"] = torch.from_numpy(stride).to(self.device)
        E = self.g.num_entries
        keys = torch.empty((E, 4), dtype=torch.int32, device=self.device)
        vals = torch.empty((E, 3), dtype=torch.float64, device=self.device)
        _lib.check(
            self.lib.apc_export_decision_vars(
                C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self.comm), self._ptr(self.flags),
                self._ptr(self._keep["export_row_base"]), self._ptr(self._keep["export_row_stride"]),
                self._ptr(keys), self._ptr(vals), self._stream()),
            "apc_export_decision_vars",
        )
        return keys, vals

    def solution_terms(self, assign: torch.Tensor):
        """assign: int16/uint16 [n_node] on the device -> (terms float64
        [n_edge, 4] = compute, comm, transition, cost of each edge's selected
        entry; slot int64[n_edge])."""
        assert self.built
        assert assign.dim() == 1 and assign.shape[0] == self.g.num_nodes and assign.is_contiguous()
        assert assign.dtype in (torch.int16, torch.uint16) and assign.device == self.comm.device
        terms = torch.empty((self.g.num_edges, 4), dtype=torch.float64, device=self.device)
        slot = torch.empty(self.g.num_edges, dtype=torch.int64, device=self.device)
        _lib.check(
            self.lib.apc_solution_terms(
                C.byref(self.problem), self._ptr(self.per_arg), self._ptr(self.comm), self._ptr(self.cost),
                self._ptr(self.flags), self._ptr(assign), self._ptr(terms), self._ptr(slot), self._stream()),
            "apc_solution_terms",
        )
        return terms, slot

    def score_random(self, seed: int, first: int, count: int) -> torch.Tensor:
        assert self.built
        out = torch.empty((count, 6), dtype=torch.float64, device=self.device)
        if self.packed_scoring and count >= _SCORE_LANES_FROM:
            return self._score_packed(None, seed, first, count, None, 0, None, out)
        return self._score_small(None, seed, first, count, None, 0, None, out)

    def score_random_window(self, seed: int, first: int, count: int, node_gid: np.ndarray, first_node: int,
                            init: Optional[torch.Tensor] = None) -> torch.Tensor:
        """score_random for a window of a larger graph (apc_score_random_window):
        draws by global node id, skips the first ``first_node`` stand-in nodes and
        continues the sums of ``init`` (the previous window's result)."""
        assert self.built
        gid = np.ascontiguousarray(node_gid, np.int32)
        assert gid.shape == (self.g.num_nodes,) and 0 <= first_node <= self.g.num_nodes
        assert init is None or (init.shape == (count, 6) and init.dtype == torch.float64 and init.is_contiguous())
        d_gid = torch.from_numpy(gid).to(self.device)
        out = torch.empty((count, 6), dtype=torch.float64, device=self.device)
        if self.packed_scoring and count >= _SCORE_LANES_FROM:
            return self._score_packed(None, seed, first, count, d_gid, first_node, init, out)
        return self._score_small(None, seed, first, count, d_gid, first_node, init, out)

    def score_window(self, assign: torch.Tensor, first_node: int, init: Optional[torch.Tensor] = None) -> torch.Tensor:
        """score() for a window of a larger graph: explicit assignments (uint16
        [n_node, n_assign], stand-in nodes included), the first ``first_node``
        nodes contribute nothing, and the sums continue from ``init``."""
        assert self.built
        assert assign.dim() == 2 and assign.shape[0] == self.g.num_nodes and assign.is_contiguous()
        assert assign.dtype in (torch.int16, torch.uint16) and assign.device == self.comm.device
        count = assign.shape[1]
        assert 0 <= first_node <= self.g.num_nodes
        assert init is None or (init.shape == (count, 6) and init.dtype == torch.float64 and init.is_contiguous())
        out = torch.empty((count, 6), dtype=torch.float64, device=self.device)
        if self.packed_scoring and count >= _SCORE_LANES_FROM:
            return self._score_packed(assign, 0, 0, count, None, first_node, init, out)
        return self._score_small(assign, 0, 0, count, None, first_node, init, out)

    def _allowed_columns(self):
        """(colbits, col_off, max_words) of apc_pack_allowed_columns for the flags as they
        are now: the layout is made once per engine, the bits on every call (one pass over
        the flags; any build or pass may have rewritten them)."""
        g = self.g
        lay = self._keep.get("column_layout")
        if lay is None:
            words = (g.edge_sdst.astype(np.int64) + 63) >> 6
            size = g.edge_ssrc.astype(np.int64) * ((words + 1) & ~1)  # a column: whole pairs of words
            own = np.ones(g.num_edges, bool) if g.edge_alias is None else g.priced
            off = np.zeros(g.num_edges, np.int64)
            off[own] = np.cumsum(size[own]) - size[own]
            if g.edge_alias is not None:  # an edge without a block of its own reads its root's columns
                off[~own] = off[g.edge_alias[~own]]
            total = int(size[own].sum())
            self._keep["column_layout_host"] = np.ascontiguousarray(off, np.int64)
            lay = self._keep["column_layout"] = (
                torch.from_numpy(off).to(self.device), max(int(words.max()) if g.num_edges else 1, 1),
                torch.empty(max(total, 1), dtype=torch.int64, device=self.device))
        d_off, max_words, colbits = lay
        _lib.check(
            self.lib.apc_pack_allowed_columns(
                C.byref(self.problem), self._ptr(self.flags), self._ptr(d_off), int(max_words), self._ptr(colbits),
                self._stream()),
            "apc_pack_allowed_columns")
        return colbits, d_off, max_words

    def _sample_tiles(self, first_node: int):
        """(apc_sample_tile records, argument rows' places, both on the device, tiles, wide, depth of the graph) of
        apc_sample_feasible_tiles for the walk from ``first_node`` on, or None: a graph such a walk does not take, or no
        layout at hand (_layout)."""
        return self._layout("sample_tiles", first_node, lambda: self._make_sample_tiles(first_node))

    def _make_sample_tiles(self, first_node: int):
        g = self.g
        n = g.num_nodes - first_node
        if n <= 0 or g.num_edges == 0 or int(g.node_nstrat[first_node:].max()) > 64:
            return None
        off, src, ssrc, nstrat = [np.ascontiguousarray(x, np.int32) for x in (
            g.node_edge_off, g.edge_src_node, g.edge_ssrc, g.node_nstrat)]
        tiles, rows, n_tile = np.empty((n, _lib.SAMPLE_TILE_BYTES), np.uint8), np.zeros(g.num_edges, np.uint8), C.c_int32(0)
        _lib.check(
            self.lib.apc_sample_tiles(
                g.num_nodes, g.num_edges, off.ctypes.data, src.ctypes.data, ssrc.ctypes.data, nstrat.ctypes.data,
                int(first_node), tiles.ctypes.data, n, rows.ctypes.data, C.byref(n_tile)),
            "apc_sample_tiles")
        if n_tile.value == 0:
            return None
        return (torch.from_numpy(tiles[:n_tile.value]).to(self.device), torch.from_numpy(rows).to(self.device),
                n_tile.value, int(nstrat[first_node:].max() > 32), int(tiles[0].view(np.int32)[_lib.SAMPLE_TILE_DEPTH]))

    def _steps_before_tiles(self, first_node: int, count: int, tiles):
        """_sample_steps where sixteen wavefronts in steps, or two on the smallest graphs, are faster than ``tiles``, else
        None."""
        n, n_edge = self.g.num_nodes - first_node, self.g.num_edges - int(self.g.node_edge_off[first_node])
        n_tile, depth = tiles[2], tiles[4]
        by_tiles = _SAMPLE_TILES_US[0] + _SAMPLE_TILES_US[1] * n + _SAMPLE_TILES_US[2] * n_tile
        step = -(-count // 16384) * (_SAMPLE_STEP_US[0] + _SAMPLE_STEP_US[1] * n_edge / n)
        if n < 6 * depth:  # two wavefronts
            two = _SAMPLE_TWO_US[1] * max(1.0, count / _SAMPLE_TWO_UP_TO)
            if _SAMPLE_TWO_US[0] + two * max(depth, n / 2) >= by_tiles:
                return None
            steps = self._sample_steps(first_node)
            return steps if steps is not None and _SAMPLE_TWO_US[0] + two * steps[1] < by_tiles else None
        if max(depth, n / 16) * step >= by_tiles:  # too many steps in any layout
            return None
        steps = self._sample_steps(first_node)
        return steps if steps is not None and steps[2] == 16 and steps[1] * step < by_tiles else None

    def _sample_steps(self, first_node: int):
        """(records on the device, steps, wavefronts) of apc_sample_feasible_steps for the walk
        from ``first_node`` on, or None: a graph such a walk does not take (columns past its
        32-bit offsets, a producer behind its consumer, more steps than nodes), or no layout at hand (_layout)."""
        return self._layout("sample_steps", first_node, lambda: self._make_sample_steps(first_node))

    def _make_sample_steps(self, first_node: int):
        g = self.g
        n = g.num_nodes - first_node
        plan = None
        if (n > 0 and g.num_edges > 0 and g.num_nodes < 1 << 24 and (g.edge_src_node < g.edge_node).all()
                and int(self._keep["column_layout_host"].max()) < 1 << 32):
            edge_off = np.ascontiguousarray(g.node_edge_off, np.int32)
            src = np.ascontiguousarray(g.edge_src_node, np.int32)
            nstrat = np.ascontiguousarray(g.node_nstrat, np.int32)
            col_off = self._keep["column_layout_host"]
            n_step, n_waves = C.c_int32(0), C.c_int32(0)
            # A node with more argument rows than a record names waits until its producers have left the
            # ring, 8 or 64 steps.  A step takes about as long as a node of the lane walk (1.2 and 1.5 us), so a
            # walk of more steps than nodes is no gain.
            recs = np.empty((n * 16, _lib.SAMPLE_REC_BYTES), np.uint8)
            rc = self.lib.apc_sample_steps(
                g.num_nodes, g.num_edges, edge_off.ctypes.data, src.ctypes.data, nstrat.ctypes.data,
                col_off.ctypes.data, int(first_node), _SAMPLE_WAVES, recs.ctypes.data, n,
                C.byref(n_step), C.byref(n_waves))
            if rc == _lib.ERR_UNSUPPORTED:
                return None
            _lib.check(rc, "apc_sample_steps")
            recs = torch.from_numpy(recs[:n_step.value * n_waves.value]).to(self.device)
            plan = (recs, n_step.value, n_waves.value)
        return plan

    def sample_feasible(self, seed: int, first: int, count: int, node_gid: Optional[np.ndarray] = None,
                        first_node: int = 0, assign: Optional[torch.Tensor] = None,
                        row_filter: Optional[dict] = None):
        """``count`` assignments drawn node by node among the strategies that select
        no forbidden (non-finite) entry against the choices made for the node's
        producers (apc_pack_allowed_columns, then apc_sample_feasible_tiles, apc_sample_steps or
        apc_sample_feasible, by strategies, batch and layout).  Returns
        (assign uint16[n_node, count] on the device, n_fallback int32[count]: nodes
        that had no such strategy and took the plain draw).  ``assign``/``first_node``:
        rows below first_node are given (a window of a larger graph); ``node_gid``:
        ids for the hashes; ``row_filter``: {node: bool per strategy}, the strategies a
        node may take at all, or "plan" for the filters feasible_plan.plan_filters makes
        for this graph (made once per engine)."""
        assert self.built
        if isinstance(row_filter, str):
            assert row_filter == "plan" and first_node == 0
            if "row_filter_plan" not in self._keep:
                from . import feasible_plan

                self._keep["row_filter_plan"] = feasible_plan.plan_filters(feasible_plan.window_masks(self.g))[0]
            row_filter = self._keep["row_filter_plan"]
        N = self.g.num_nodes
        if assign is None:
            assert first_node == 0
            assign = torch.empty((N, count), dtype=torch.uint16, device=self.device)
        assert assign.shape == (N, count) and assign.dtype == torch.uint16 and assign.is_contiguous()
        d_gid = None
        if node_gid is not None:
            d_gid = torch.from_numpy(np.ascontiguousarray(node_gid, np.int32)).to(self.device)
        fallback = torch.empty(count, dtype=torch.int32, device=self.device)
        colbits, d_off, _ = self._allowed_columns()
        d_keep = d_keep_off = None
        if row_filter:
            # bit out_idx mod 64 of word out_idx / 64, the words of the filtered nodes one after the other
            keep_off = np.full(N, -1, np.int64)
            words = []
            at = 0
            for v in sorted(row_filter):
                keep = np.asarray(row_filter[v], bool)
                assert keep.shape == (int(self.g.node_nstrat[v]),)
                padded = np.zeros(-(-keep.shape[0] // 64) * 64, np.uint8)
                padded[: keep.shape[0]] = keep
                w = np.packbits(padded, bitorder="little").view(np.uint64)
                keep_off[v] = at
                at += w.shape[0]
                words.append(w)
            d_keep = torch.from_numpy(np.concatenate(words).view(np.int64)).to(self.device)
            d_keep_off = torch.from_numpy(keep_off).to(self.device)
        tiles = self._sample_tiles(first_node) if _SAMPLE_TILES and not _SAMPLE_WAVES and count > 0 else None
        steps = scratch = None
        if tiles is not None:
            steps = self._steps_before_tiles(first_node, count, tiles)
            if steps is None:
                scratch = self._scratch((tiles[2] + 1) * _lib.SAMPLE_IMAGE_BYTES)
        if scratch is not None:
            d_tiles, d_rows, n_tile, wide, _ = tiles
            _lib.check(
                self.lib.apc_sample_feasible_tiles(
                    C.byref(self.problem), self._ptr(d_tiles), n_tile, self._ptr(d_rows), self._ptr(colbits),
                    self._ptr(d_off), self._ptr(scratch), int(seed), int(first), int(count), self._ptr(d_gid),
                    self._ptr(d_keep), self._ptr(d_keep_off), wide, self._ptr(assign), self._ptr(fallback), self._stream()),
                "apc_sample_feasible_tiles")
            self.last_sample_backend = "tiles"
            return assign, fallback
        if steps is None and count < max(_SAMPLE_LANES_FROM.values()):
            steps = self._sample_steps(first_node)
        if steps is not None and count < _SAMPLE_LANES_FROM[steps[2]]:
            recs, n_step, n_waves = steps
            _lib.check(
                self.lib.apc_sample_feasible_steps(
                    C.byref(self.problem), self._ptr(recs), n_step, n_waves, self._ptr(colbits), self._ptr(d_off),
                    int(seed), int(first), int(count), self._ptr(d_gid), self._ptr(d_keep), self._ptr(d_keep_off),
                    self._ptr(assign), self._ptr(fallback), self._stream()),
                "apc_sample_feasible_steps")
            self.last_sample_backend = "steps"
            return assign, fallback
        _lib.check(
            self.lib.apc_sample_feasible(
                C.byref(self.problem), self._ptr(colbits), self._ptr(d_off), int(seed), int(first), int(count),
                self._ptr(d_gid), int(first_node), self._ptr(d_keep), self._ptr(d_keep_off), self._ptr(assign),
                self._ptr(fallback), self._stream()),
            "apc_sample_feasible")
        self.last_sample_backend = "lanes"
        return assign, fallback

    def random_assignment(self, seed: int, a: int) -> np.ndarray:
        """The out_idx per node that score_random draws for assignment a."""
        g = self.g
        return np.asarray(
            [self.lib.apc_random_assignment(int(seed), int(a), v, int(g.node_nstrat[v])) for v in range(g.num_nodes)],
            dtype=np.int64,
        )

    # -- results on host --------------------------------------------------------
    def compact_entries(self):
        """(comm, cost, flags) on the device with one element per decision variable:
        the entry arrays without the padding between edge blocks
        (apc_compact_entries), in the order of the ILP's columns."""
        assert self.built
        g = self.g
        if "var_start" not in self._keep:
            start = np.zeros(g.num_edges + 1, np.int64)
            np.cumsum(g.block_sizes(), out=start[1:])
            self._keep["var_start"] = torch.from_numpy(start).to(self.device)
        E = g.num_entries
        comm = torch.empty(E, dtype=torch.float64, device=self.device)
        cost = torch.empty(E, dtype=torch.float64, device=self.device)
        flags = torch.empty(E, dtype=torch.uint8, device=self.device)
        _lib.check(
            self.lib.apc_compact_entries(
                C.byref(self.problem), self._ptr(self._keep["var_start"]), self._ptr(self.comm), self._ptr(self.cost),
                self._ptr(self.flags), self._ptr(comm), self._ptr(cost), self._ptr(flags), self._stream()),
            "apc_compact_entries")
        return comm, cost, flags

    def results(self, compact: bool = False) -> Dict[str, np.ndarray]:
        """The five result arrays on the host.  ``compact``: comm, cost and flags
        per decision variable (padding taken out on the device) instead of per
        slot.  They are copied into pinned memory (torch keeps freed pinned
        blocks, so only a process's first call pays for pinning) by copies that
        run back to back; the arrays returned own it."""
        self.check_status()
        src = {name: getattr(self, name) for name in ("comm", "cost", "flags", "compute", "per_arg")}
        if compact and self.g.num_slots != self.g.num_entries:
            src["comm"], src["cost"], src["flags"] = self.compact_entries()
        out = {}
        for name, t in src.items():
            dst = torch.empty(t.shape, dtype=t.dtype, pin_memory=_READBACK_PINNED)
            dst.copy_(t, non_blocking=_READBACK_PINNED)
            out[name] = dst
        torch.cuda.current_stream(self.device).synchronize()
        return {k: v.numpy() for k, v in out.items()}
