"""Dense trellis layers for decode: every matrix of one vLLM layer in as few esp_dense launches as the codes allow (the
interface of vllm_espalier/dense.py: Dense, plan, scratch, MAX_ROWS).

A vLLM layer fuses several checkpoint matrices (q/k/v, gate/up); each keeps its own suh/svh, so they are never
concatenated into one trellis. A launch takes up to four of them that share the input width, the bit width and the
codebook; it reads x once in the model's dtype and writes each matrix's columns of y in that dtype. Up to MAX_ROWS rows
a launch; ops.py windows longer inputs.

The K split of a launch (`plan`) is a function of the layer's shape alone, so the bits of a row never depend on the
other rows of the batch.
"""
from __future__ import annotations

import itertools
import os
from dataclasses import dataclass, field

import torch

from ._env import env
from ._streams import hand_out, raw_stream
from .experts import KERNEL_CB, ext

MAX_ROWS = 32
COUNTER_STRIDE = 32          # ints between two 128-column blocks' arrival counters (one 128-byte line each)
MAX_MATRICES = 4             # matrices one esp_dense launch takes
ROT_SMEM = int(os.environ.get("ESPALIER_DENSE_ROTATION_SMEM", 64 * 1024))   # fuse the input rotation up to this much LDS


def plan(K: int, N: int, sms: int) -> tuple[int, int, int]:
    """(K splits SK, waves a workgroup W, tiles in flight) for a K -> N layer of 128-column blocks, from its shape
    alone so a row's bits never depend on the batch (the reference's sm89 heuristic is dense.py:22-39). A gfx950
    workgroup is 4 * KW waves on one block, KW of them on every 32-k step column; a split is a run of whole 32-k
    steps, SK need not divide them. The decode of a workgroup's share is bound by its CU's VALU, so the plan spreads
    the layer over the CUs, SK = CUs // blocks (one workgroup a CU), but keeps 4 steps a split: below that the
    fixed costs (rotation, hand-off) outweigh the shorter decode, and 32-row windows lose more to the extra partials
    than single rows gain. Then 16 waves when a split has 4 steps or more, else 4, but at most 8 when the launch has
    more workgroups than CUs (the LM head: 97 us against 113 at 16 waves). bench.py --sweep (cold, MI355X) confirms the
    K splits of config 2's four launches at 1 and 32 rows, and the 16 waves also for the 4-step splits of the shared
    gate/up and down (1 row 6.95 -> 6.91 and 6.49 -> 6.46 us, 32 rows 12.1 -> 10.2 and 8.7 -> 8.0 us against 8
    waves). ESPALIER_DENSE_TILE_PLAN="sk,w,pf" forces."""
    forced = env("ESPALIER_DENSE_TILE_PLAN")
    if forced:
        sk, w, pf = (int(v) for v in forced.split(","))
        return sk, w, pf
    nb = N // 128
    steps_all = K // 32
    sk = max(1, min(steps_all // 4, sms // nb))
    steps = -(-steps_all // sk)
    w = 16 if steps >= 4 else 4
    if nb * sk > sms:
        w = min(w, 8)            # more workgroups than CUs: two of 8 waves share a CU and hide each other's waits
    return sk, w, 2


def tile_plan(K: int, N: int) -> int:
    """K splits of a prompt launch (esp_dense_tile) of a K -> N layer, from its shape alone (so a row's bits never
    depend on the prompt's length): the most splits that keep a 512-row prompt (4 tiles of 128 rows) within two 8-wave
    workgroups a CU, 4 * blocks * SK <= 512, so the grid stays resident and the split-K finish is spread over the
    splits; at most 8 (the spread finish's batch of partial loads) and splits of at least 128 k. From a sweep of every
    launch's SK at 128 / 512 / 2048 rows with the spread finish (config 2: qkv 3, o 8, shared gate/up 8, shared down 4,
    the fastest at 512 and 128 rows: o 35.7 -> 31.8 us and shared down 20.9 -> 17.4 us at 512 rows against the earlier
    4 and 1). At 2048 rows, where the grid is not resident and one split finishes each tile, fewer splits would be
    faster (o 81 us at 2 against 109 at 8). ESPALIER_DENSE_PROMPT_SK forces."""
    forced = env("ESPALIER_DENSE_PROMPT_SK")
    if forced:
        return int(forced)
    blocks = N // 128
    return max(1, min(128 // blocks, 8, K // 128))


def prompt_rows(K: int, N: int) -> int:
    """Rows from which a prompt through a K -> N launch runs as esp_dense_prompt (2 launches, each weight decoded once)
    instead of windows of MAX_ROWS rows, with the same bits. Four windows (97 rows) for most shapes: config 2's four layers
    together 114 us against 181 at 128 rows, 4096 -> 2048 42 against 45 at 97. But the prompt GEMM walks K in a line, about
    7 us a 1024 k where its few workgroups do not hide it, while a window's time hardly grows with K (its K splits fill the
    CUs): past K = 4096 a layer of 512 to 2048 columns takes one window more for each 4096 k (MI355X, windows against prompt:
    8192 -> 2048 56 / 72 us and 69 / 67 at 97 and 129 rows, 12288 -> 1024 86 / 91 and 103 / 91 at 160 and 192, 16384 -> 1024
    111 / 114 and 130 / 114 at 192 and 224; 8192 -> 4096 68 / 66 and 16384 -> 256 1.05 at 97)."""
    if K <= 4096 or N > 2048 or N < 512 or (N < 1024 and K <= 8192):
        return PROMPT_MIN_ROWS
    return PROMPT_MIN_ROWS + MAX_ROWS * -(-(K - 4096) // 4096)


TILE_ROWS = 128              # rows a prompt-launch workgroup
TILE_SLOTS = 2               # k slots a workgroup of esp_dense_tile
PROMPT_MIN_ROWS = 97         # rows from which prompt_rows sends a prompt to esp_dense_prompt at the earliest
PROMPT_ROWS = 4096           # rows one esp_dense_prompt call takes (bounds its scratch)
PROMPT_WEIGHTS = 1 << 27     # weights a launch decodes whole (2 bytes each)
# launches whose last K split can poll the others' partials run as esp_dense_own over an all-ones partials buffer (the
# same bits, no arrival count); ESPALIER_DENSE_OWN=0 runs every launch as esp_dense
OWN = env("ESPALIER_DENSE_OWN", "1") != "0"


STREAM_MAX_ROWS = 6          # rows of esp_dense_stream (2 with the norm inside)
STREAM_WAIT_US = 200         # a workgroup's wait for its predecessor's sums before it makes them itself (the whole launch takes less)
STREAM_PARTS = 16            # HIP streams of which a layer keeps a hand-off buffer (3 MiB)
STREAM_SPARES = 8            # captured launches that get one; more run as esp_dense (a fill in the graph would take 6 us)
# wide launches over a few rows run as esp_dense_stream (the same bits); ESPALIER_DENSE_STREAM=0 runs them as esp_dense
STREAM = env("ESPALIER_DENSE_STREAM", "1") != "0"


class _SharedScratch:
    """The split-K partials Z (fp32) and the unfused rotation's rows xh (fp16), one pair a device, shared by every
    layer (layers run one after another). Sizes only grow. A pair that a growth replaces is kept for good only when a
    graph may write to it (it was handed out during a stream capture); otherwise it is dropped, and the caching
    allocator reuses its memory once every stream that it was handed out on is done with it, so a series of growing
    prompts outside capture keeps only the current pair."""

    def __init__(self, fill=None, dtype=torch.float32):
        self.fill, self.dtype = fill, dtype  # Z's 32-bit words to begin with (None: any), and its type
        self.current: dict = {}
        self.captured: set = set()          # devices whose current pair was handed out during a capture
        self.streams: dict = {}             # device -> streams that its current pair was handed out on
        self.retired: list = []

    def reserve(self, device, z_floats: int, xh_halves: int):
        have = self.current.get(device)
        capturing = device.type == "cuda" and torch.cuda.is_current_stream_capturing()
        if have is not None and have[0].numel() >= z_floats and have[1].numel() >= xh_halves:
            if capturing:
                self.captured.add(device)
            elif (raw := raw_stream(device)) not in self.streams[device]:
                hand_out(have, self.streams[device], device, raw)
            return have
        if have is not None:
            if device in self.captured:
                self.retired.append(have)
            z_floats, xh_halves = max(z_floats, have[0].numel()), max(xh_halves, have[1].numel())
        self.captured.discard(device)
        z = torch.empty(max(z_floats, 1), dtype=torch.int32, device=device)
        if self.fill is not None:
            z.fill_(self.fill)
        pair = (z.view(self.dtype), torch.empty(max(xh_halves, 1), dtype=torch.float16, device=device))
        self.current[device] = pair
        self.streams[device] = {raw_stream(device)}
        if capturing:
            self.captured.add(device)
        return pair


_SHARED = _SharedScratch()
_OWN = _SharedScratch(fill=-1)               # all-ones partials (esp_dense_own)


def scratch(device, z_floats: int, xh_halves: int):
    """(Z, xh) of the device, grown to at least the given sizes."""
    return _SHARED.reserve(device, z_floats, xh_halves)


def own_partials(device, z_floats: int):
    """The device's all-ones partials buffer of esp_dense_own (left all-ones by every launch), grown to at least
    z_floats."""
    return _OWN.reserve(device, z_floats, 0)[0]


def restore_own_partials() -> None:
    """Every all-ones partials buffer, those that graphs hold too, all-ones again (after a wait that gave up; nothing may be
    running)."""
    for z, _ in [*_OWN.current.values(), *_OWN.retired]:
        z.view(torch.int32).fill_(-1)


def polls(M: int, sk: int, w: int) -> bool:
    """Whether a launch of M rows, sk K splits and w waves takes esp_dense_own's polled hand-off: its last split holds
    one (row, split) partial a 32-lane half."""
    return sk > 1 and M * (sk - 1) <= 2 * w


_PROMPT = _SharedScratch()
_PROMPT_COUNTERS = _SharedScratch(fill=0, dtype=torch.int32)


def prompt_scratch(device, z_floats: int, xh_halves: int, counters: int):
    """(Z, xh, counters) of the device for prompt launches, grown to at least the given sizes (the counters zero, and
    left zero by every launch)."""
    return *_PROMPT.reserve(device, z_floats, xh_halves), _PROMPT_COUNTERS.reserve(device, counters, 0)[0]


def _cu_count(device) -> int:
    if device.type == "cuda" and torch.cuda.is_available():
        return torch.cuda.get_device_properties(device).multi_processor_count
    return 256                                   # MI355X


@dataclass(frozen=True)
class Launch:
    """One esp_dense launch: the matrices (indices into Dense.mats), their common half-bits and kernel codebook, the
    columns they write, and the shape's plan."""
    members: tuple
    k2: int
    cb: int
    n: int
    sk: int
    w: int
    pf: int
    stream: range = field(default=range(0), compare=False)      # rows that run as esp_dense_stream (stream_rows)


def stream_rows(K: int, n: int, k2: int, matrices: int, sk: int, w: int, cus: int) -> range:
    """Rows over which a launch runs as esp_dense_stream: one matrix of more column blocks than CUs in one K split (an LM
    head), and rows that leave two workgroups a CU. 2048 -> 151936, graph replays: 6 bits (mcg) 73.1 us as a workgroup a block
    and 66.1 streamed at one row, 76.8 and 67.9 at four; 4 bits (int6) 77.7 and 73.2, 106.9 and 76.4. At 2 bits a block is
    decoded too soon for the shares to pay below four rows (2048 -> 128000, e2m1, at one and four rows 61 and 63 us, 82 and
    64), at one bit at none (42 and 45); nor do they in a block of one or two stages, but where the blocks' last round of
    workgroups is long (512 -> 76800, int6 4 bits: 17.1 and 17.4 us; 512 -> 151936, mcg: 1.04 to 1.12)."""
    blocks = n // 128
    if not (matrices == 1 and sk == 1 and w == 4 * TILE_SLOTS and K % 256 == 0 and K * n <= 1 << 33 and n < 1 << 24 and
            blocks > cus and k2 >= 4 and (K >= 768 or blocks > 4 * cus)):
        return range(0)
    fit = (80 * 1024 - 512 - 4096 * k2) // (2 * K + 16 + 1024)
    return range(4 if k2 == 4 else 1, min(fit, STREAM_MAX_ROWS) + 1)


class Dense:
    MAX_ROWS = MAX_ROWS

    def __init__(self, mats, n_out: int | None = None):
        self.mats = list(mats)
        widths = {m.in_features for m in self.mats}
        if len(widths) != 1:
            raise ValueError(f"the matrices of a dense layer must share their input width, got {sorted(widths)}")
        (self.K,) = widths
        offsets = list(itertools.accumulate((m.out_features for m in self.mats), initial=0))
        self.col0, self.N = offsets[:-1], offsets[-1]
        self.n_out = n_out or self.N
        device = self.mats[0].trellis.device
        self.cus = cus = _cu_count(device)
        self.launches = []
        for code, run in itertools.groupby(range(len(self.mats)), key=self._code):
            run = list(run)
            for i in range(0, len(run), MAX_MATRICES):
                members = tuple(run[i:i + MAX_MATRICES])
                n = sum(self.mats[j].out_features for j in members)
                self.launches.append(self._launch(members, *code, n, *plan(self.K, n, cus)))
        self.prompt_rows = max(prompt_rows(self.K, l.n) for l in self.launches)
        blocks = max(l.n // 128 for l in self.launches)
        self.counters = torch.zeros(COUNTER_STRIDE * blocks, dtype=torch.int32, device=device)
        scratch(device, max(l.sk * MAX_ROWS * l.n for l in self.launches), 4 * MAX_ROWS * self.K)
        own_partials(device, max(l.sk * 2 * l.w // max(l.sk - 1, 1) * l.n for l in self.launches))
        # esp_dense_stream's hand-off buffers: a HIP stream's own, spare ones for captured launches, and those in graphs
        self._stream_parts, self._stream_graphs = {}, []
        streams = any(l.stream for l in self.launches)
        self._stream_spare = list(self._new_parts(device, STREAM_SPARES)) if streams else []

    def _launch(self, members, k2, cb, n, sk, w, pf) -> Launch:
        return Launch(members, k2, cb, n, sk, w, pf, stream_rows(self.K, n, k2, len(members), sk, w, self.cus))

    def _code(self, i: int) -> tuple[int, int]:
        m = self.mats[i]
        return 2 * m.K, KERNEL_CB[m.cb]

    @property
    def groups(self) -> list:
        """(matrix indices, k2, kernel codebook) of each launch."""
        return [(list(l.members), l.k2, l.cb) for l in self.launches]

    @property
    def plans(self) -> list:
        """(SK, W, PF) of each launch."""
        return [(l.sk, l.w, l.pf) for l in self.launches]

    @plans.setter
    def plans(self, plans) -> None:
        """Replace the launches' plans (the scratch must already be large enough for them)."""
        if len(plans) != len(self.launches):
            raise ValueError(f"{len(plans)} plans for {len(self.launches)} launches")
        self.launches = [self._launch(l.members, l.k2, l.cb, l.n, *p) for l, p in zip(self.launches, plans)]

    def forward(self, x, trellis=None, suh=None, svh=None, out=None):
        """x [M, K] (M <= MAX_ROWS) -> [M, n_out] in x's dtype. trellis / suh / svh: lists that replace the matrices'
        own tensors (the module buffers a compiled graph passes in)."""
        codes = trellis or [m.trellis for m in self.mats]
        pre = suh or [m.suh for m in self.mats]
        post = svh or [m.svh for m in self.mats]
        y = torch.empty((x.shape[0], self.n_out), dtype=x.dtype, device=x.device) if out is None else out
        if self.n_out > self.N:
            y[:, self.N:].zero_()                     # padding columns (the LM head's vocabulary padding)
        if x.stride(-1) != 1:
            x = x.contiguous()
        for l in self.launches:
            self._window(x, codes, pre, post, y, l)
        return y

    def _streams(self, M: int, l) -> bool:
        """Whether launch l over M rows runs as esp_dense_stream (its plan's bits)."""
        return STREAM and M in l.stream

    def _new_parts(self, device, n: int):
        floats = 2 * _cu_count(device) * (256 * STREAM_MAX_ROWS + COUNTER_STRIDE)
        return torch.full((n, floats), -1, dtype=torch.int32, device=device).view(torch.float32).unbind()

    def _stream_part(self, device):
        """The all-ones hand-off buffer for an esp_dense_stream launch on the current HIP stream, left all-ones by every
        launch: launches on one stream run one after another, and no two streams share one. A captured launch has one of
        its own, since a graph replays on any stream, kept with the layer. None past STREAM_PARTS streams or STREAM_SPARES
        captured launches."""
        if torch.cuda.is_current_stream_capturing():
            try:
                part = self._stream_spare.pop()
            except IndexError:
                return None
            self._stream_graphs.append(part)
            return part
        key = torch.cuda.current_stream(device).cuda_stream
        part = self._stream_parts.get(key)
        if part is None and len(self._stream_parts) < STREAM_PARTS:
            part = self._stream_parts.setdefault(key, self._new_parts(device, 1)[0])
        return part

    def _window(self, x, codes, pre, post, y, l) -> None:
        """Launch l over the rows of x (at most MAX_ROWS) into its columns of y."""
        if x.shape[0] in l.stream and STREAM and (part := self._stream_part(x.device)) is not None:
            i = l.members[0]
            ext().dense_stream(x, None, None, None, 0.0, None, codes[i], pre[i], post[i], self.col0[i], y, part,
                               STREAM_WAIT_US, l.k2, l.cb)
            return
        z, xh = scratch(x.device, 0, 0)
        e = ext()
        M = x.shape[0]
        pick = l.members
        # a launch whose last split can poll the others' partials runs over the all-ones buffer (the same bits)
        if OWN and polls(M, l.sk, l.w):
            run, zl = e.dense_own, own_partials(x.device, l.sk * M * l.n)
        else:
            run, zl = e.dense, z
        run(x, [codes[i] for i in pick], [pre[i] for i in pick], [post[i] for i in pick], [self.col0[i] for i in pick],
            y, xh, zl, self.counters, l.k2, l.cb, l.sk, l.w, l.pf, ROT_SMEM)

    def prompts(self) -> bool:
        """Whether forward_prompt takes this layer: 128-wide blocks, and no launch with too many weights to decode
        whole or with a K split shorter than its k slots."""
        return (self.K % 128 == 0 and all(m.out_features % 128 == 0 for m in self.mats) and
                all(self.K * l.n <= PROMPT_WEIGHTS and l.sk * (l.w // 4) <= self.K // 32 for l in self.launches))

    def _tile_is_window(self, T: int, launch, sk: int | None = None) -> bool:
        """Whether T rows of a launch in the tile mode run as one decode launch, whose sums are then esp_dense_tile's: no
        K split and two k slots (the LM head, whose last row a prompt takes: 125 us as a 128-row tile, 72 as a window).
        sk: its tile_plan, where the caller has it."""
        return (T <= MAX_ROWS and launch.sk == 1 and launch.w == 4 * TILE_SLOTS and
                (tile_plan(self.K, launch.n) if sk is None else sk) == 1)

    def _tile_decodes_once(self, T: int, launch, sk: int | None = None) -> bool:
        """Whether T rows of a launch in the tile mode run as esp_dense_prompt (the bits of esp_dense_tile, every weight
        decoded once): where esp_dense_tile's grid is past two 8-wave workgroups a CU, so its tiles decode the weights
        again in a second round and its splits' partials follow one another (2048 -> 5120 at 509 / 1024 / 2048 rows: 40
        / 70 / 125 us against 38 / 48 / 76; 4096 -> 2048: 33 / 59 / 105 against 41 / 42 / 57). The second round has to cost
        something, so the line lies later (MI355X, tile against prompt, us):
          a last tile of up to 32 rows costs next to nothing: from K = 4096, and for the mcg weights (cheaper to decode) of
          large layers, it is not counted (8192 -> 2048 at 520 rows 52 / 60, 12288 -> 4096 of int6 123 / 126);
          mcg below 8 bits: 800 workgroups from K = 12288 (12288 -> 4096 at 768 / 900 rows 134 / 139 and 165 / 147), 1000
          from 192 column blocks (4096 -> 24576 at 512 / 700 rows 163 / 168 and 232 / 224), 640 for up to 2048 columns from
          K = 8192 (8192 -> 2048 of 2 bits at 576 / 700 rows 56 / 61 and 62 / 61)."""
        sk = tile_plan(self.K, launch.n) if sk is None else sk
        K, blocks = self.K, launch.n // 128
        cheap = launch.cb == KERNEL_CB[0] and launch.k2 < 16
        uncounted = 32 if K >= 4096 or (cheap and K * launch.n >= 1 << 24) else 0
        limit = 512
        if cheap:
            limit = 800 if K >= 12288 else 1000 if blocks >= 192 else 640 if K >= 8192 and blocks <= 16 else 512
        return (-(-max(T - uncounted, 0) // TILE_ROWS) * blocks * sk > limit and K * launch.n <= PROMPT_WEIGHTS and
                sk * TILE_SLOTS <= K // 32)

    def _prompt(self, x, codes, pre, post, y, launch, sk: int, slots: int) -> None:
        pick = launch.members
        for r0 in range(0, x.shape[0], PROMPT_ROWS):
            rows = slice(r0, r0 + PROMPT_ROWS)
            ext().dense_prompt(x[rows], [codes[i] for i in pick], [pre[i] for i in pick], [post[i] for i in pick],
                               [self.col0[i] for i in pick], y[rows], launch.k2, launch.cb, sk, slots)

    def forward_prompt(self, x, trellis=None, suh=None, svh=None, out=None):
        """x [T, K], any T (a prompt) -> [T, n_out] in x's dtype, with forward's bits a row and every weight decoded once
        (esp_dense_prompt; only when prompts()). trellis / suh / svh as in forward."""
        codes = trellis or [m.trellis for m in self.mats]
        pre = suh or [m.suh for m in self.mats]
        post = svh or [m.svh for m in self.mats]
        y = torch.empty((x.shape[0], self.n_out), dtype=x.dtype, device=x.device) if out is None else out
        if self.n_out > self.N:
            y[:, self.N:].zero_()
        if x.stride(-1) != 1:
            x = x.contiguous()
        for l in self.launches:
            self._prompt(x, codes, pre, post, y, l, l.sk, l.w // 4)
        return y

    def _tiles(self, T: int) -> list:
        """(launch, its K splits, how it runs over T rows in the tile mode: "tile", "window" or "once") of every launch."""
        runs = []
        for l in self.launches:
            sk = tile_plan(self.K, l.n)
            runs.append((l, sk, "window" if self._tile_is_window(T, l, sk) else
                         "once" if self._tile_decodes_once(T, l, sk) else "tile"))
        return runs

    def _reserve_tiles(self, T: int, runs, device):
        """(Z, xh, counters) for the launches of `runs` that run as esp_dense_tile, or None when none does."""
        tiles = -(-T // TILE_ROWS)
        z = xh = cnt = 0
        for l, sk, how in runs:
            if how == "tile":
                z = max(z, tiles * sk * TILE_ROWS * l.n)
                xh = max(xh, len(l.members) * -(-T // 16) * 16 * self.K)
                cnt = max(cnt, tiles * (l.n // 128) * COUNTER_STRIDE)
        return prompt_scratch(device, z, xh, cnt) if z else None

    def reserve_prompt(self, T: int) -> None:
        """Grow the prompt scratch for forward_tile over T rows (done before a graph is captured); launches that run as
        decode launches or as esp_dense_prompt there need none."""
        self._reserve_tiles(T, self._tiles(T), self.mats[0].trellis.device)

    def forward_tile(self, x, trellis=None, suh=None, svh=None, out=None):
        """x [T, K], any T (a prompt) -> [T, n_out] in x's dtype, each weight decoded once for every 128 rows
        (esp_dense_tile) or once (esp_dense_prompt, the same bits). A row's bits are its own (the same at any T), not
        those of forward. trellis / suh / svh: lists that replace the matrices' own tensors, as in forward."""
        codes = trellis or [m.trellis for m in self.mats]
        pre = suh or [m.suh for m in self.mats]
        post = svh or [m.svh for m in self.mats]
        T = x.shape[0]
        y = torch.empty((T, self.n_out), dtype=x.dtype, device=x.device) if out is None else out
        if self.n_out > self.N:
            y[:, self.N:].zero_()
        if x.stride(-1) != 1:
            x = x.contiguous()
        runs = self._tiles(T)
        scratch_tile = self._reserve_tiles(T, runs, x.device)
        for l, sk, how in runs:
            if how == "window":
                self._window(x, codes, pre, post, y, l)
            elif how == "once":
                self._prompt(x, codes, pre, post, y, l, sk, TILE_SLOTS)
            else:
                z, xh, cnt = scratch_tile
                pick = l.members
                ext().dense_tile(x, [codes[i] for i in pick], [pre[i] for i in pick], [post[i] for i in pick],
                                 [self.col0[i] for i in pick], y, xh, z, cnt, l.k2, l.cb, sk)
        return y

    def norm_fusable(self, M: int) -> bool:
        """Whether forward_rmsnorm runs in one launch for M rows: a single launch, four waves a row, and the rotated
        rows within the fused rotation's shared memory."""
        if len(self.launches) != 1:
            return False
        l = self.launches[0]
        steps = -(-(self.K // 32) // l.sk)
        blocks = -(-(steps * 32 + 96) // 128)
        return M <= l.w // 4 and self.K <= 8192 and M * blocks * 128 * 2 <= ROT_SMEM

    def forward_rmsnorm(self, h, d1, d2, norm_w, eps: float, h_out, out):
        """forward(RMSNorm(h + d1 + d2) * norm_w) with the residual h + d1 + d2 stored to h_out, the norm made inside
        the launch (bit-identical to add_rmsnorm then forward). h, d1, d2: [M, K] contiguous, the model's dtype."""
        l = self.launches[0]
        ms = [self.mats[i] for i in l.members]
        if self._streams(h.shape[0], l) and (part := self._stream_part(h.device)) is not None:
            m = ms[0]
            ext().dense_stream(h, d1, d2, norm_w, eps, h_out, m.trellis, m.suh, m.svh, self.col0[l.members[0]], out,
                               part, STREAM_WAIT_US, l.k2, l.cb)
            return out
        z, _ = scratch(h.device, 0, 0)
        ext().dense_rmsnorm(h, d1, d2, norm_w, eps, h_out, [m.trellis for m in ms], [m.suh for m in ms],
                            [m.svh for m in ms], [self.col0[i] for i in l.members], out, z, self.counters, l.k2, l.cb,
                            l.sk, l.w, ROT_SMEM)
        return out


class DenseMulti:
    """Several one-launch Dense layers as a single esp_dense_multi launch: independent layers side by side, or a chain
    in which layer i reads layer i-1's output (after[i]): one launch gap and one weight-landing latency for all of
    them. Every layer keeps its own plan's K splits; the waves a workgroup are the same for all (W), so a layer's bits
    equal its own launch at that W."""

    def __init__(self, layers, after=None, W: int = 16):
        self.layers = list(layers)
        self.after = list(after) if after is not None else [False] * len(self.layers)
        if not 1 <= len(self.layers) <= 4 or len(self.after) != len(self.layers) or self.after[0]:
            raise ValueError("1 to 4 layers; only a layer after the first may read the previous one's output")
        if any(len(d.launches) != 1 for d in self.layers):
            raise ValueError("every layer of a multi launch must be a single launch group")
        self.W = W
        # a chain's hand-off maps a consumer's ticket to a launch through its K splits, over counts that only grow: the
        # plans are fixed here, and forward refuses a layer whose plan has changed since
        self.plans = [d.launches[0] for d in self.layers]
        device = self.layers[0].mats[0].trellis.device
        blocks = sum(d.launches[0].n // 128 for d in self.layers)
        # the split-K arrival counters (left zero by every launch), then a chain's 64-bit running hand-off counts (a
        # column block's done count and its ticket count)
        self.split_counters = COUNTER_STRIDE * blocks
        self.counters = torch.zeros(3 * self.split_counters, dtype=torch.int32, device=device)
        z = sum(-(-(d.launches[0].sk * MAX_ROWS * d.launches[0].n) // 64) * 64 for d in self.layers)
        scratch(device, z, 0)

    def forward(self, xs, outs, norm=None):
        """xs[i] [M, K_i] rows of layer i (for a layer after its predecessor, a view of that layer's output); outs[i]
        [M, n_out_i] in the model's dtype. norm = (h, d1, d2, w, eps, h_out): layer 0's rows are RMSNorm(h + d1 + d2)
        * w, made in the launch, with the residual stored to h_out (xs[0] is then unused)."""
        z, _ = scratch(outs[0].device, 0, 0)
        launches = [d.launches[0] for d in self.layers]
        if launches != self.plans:
            raise ValueError("a layer's plan changed after its multi launch was built: build a new DenseMulti")
        h, d1, d2, w, eps, h_out = norm if norm is not None else (None, None, None, None, 0.0, None)
        x0 = h if norm is not None else xs[0]
        ext().dense_multi([x0] + list(xs[1:]), [[d.mats[i].trellis for i in l.members] for d, l in zip(self.layers, launches)],
                          [[d.mats[i].suh for i in l.members] for d, l in zip(self.layers, launches)],
                          [[d.mats[i].svh for i in l.members] for d, l in zip(self.layers, launches)],
                          [[d.col0[i] for i in l.members] for d, l in zip(self.layers, launches)], list(outs),
                          [l.k2 for l in launches], [l.cb for l in launches], [l.sk for l in launches],
                          [int(a) for a in self.after], z, self.counters, self.W, ROT_SMEM, h, d1, d2, w, h_out, eps)
        return outs
