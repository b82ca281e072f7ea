"""GEMM dispatch policy (mxllm/ops/gemm.py) on CPU: the measured-win table and the persistent-kernel
guard for multi-rank runs."""
import os
import socket
import subprocess
import sys

import pytest
import torch
import torch.multiprocessing as mp

import mxllm.ops  # noqa: F401
from mxllm.ops import gemm


def _persistent_entry():
    for key, ph in gemm._table().items():
        if ph == 5:
            return key
    pytest.skip("no persistent (ph 5) entry in the tuning table")


def test_table_has_persistent_fp32_dw_entries():
    form, M, N, K, out = _persistent_entry()
    assert form == "tt" and out == "f32"
    assert gemm.schedule(form, M, N, K, torch.float32) == 5  # world 1: the persistent kernel


def _worker(rank, world, port, key, q):
    os.environ.update(MASTER_ADDR="127.0.0.1", MASTER_PORT=str(port))
    import torch.distributed as dist

    dist.init_process_group("gloo", rank=rank, world_size=world)
    from mxllm.ops import gemm as g

    form, M, N, K, _ = key
    q.put((rank, g.schedule(form, M, N, K, torch.float32)))
    dist.destroy_process_group()


def test_persistent_gemm_is_world1_only():
    """In a group of > 1 ranks the persistent shapes fall back to the one-tile-per-workgroup 4-phase
    launch (collective kernels holding CUs would stall the fixed tile shares)."""
    key = _persistent_entry()
    with socket.socket() as s:
        s.bind(("127.0.0.1", 0))
        port = s.getsockname()[1]
    ctx = mp.get_context("spawn")
    q = ctx.Queue()
    ps = [ctx.Process(target=_worker, args=(r, 2, port, key, q)) for r in range(2)]
    for p in ps:
        p.start()
    got = dict(q.get(timeout=120) for _ in range(2))
    for p in ps:
        p.join(60)
        assert p.exitcode == 0
    assert got == {0: 4, 1: 4}


@pytest.mark.parametrize("env,rows,norm_rows", [({}, 32, 4), ({"MXLLM_SKINNY_M": "0"}, 0, 0), ({"MXLLM_SKINNY_M": "3"}, 3, 3),
                                                ({"MXLLM_SKINNY_M": "16"}, 16, 4), ({"MXLLM_NORM_FUSED_M": "1"}, 32, 1),
                                                ({"MXLLM_NORM_FUSED_M": "0"}, 32, 0)])
def test_switches_bound_every_decode_gemm(env, rows, norm_rows):
    """MXLLM_SKINNY_M and MXLLM_NORM_FUSED_M are upper limits for the rows of all decode kernels where they are set."""
    code = ("import sys; import mxllm.ops; m = sys.modules['mxllm.ops.linear']; r = range(1, 40); "
            "print(max([M for M in r if m._stream_fits(M, 2048)], default=0), "
            "max([M for M in r if m._norm_stream(M, 2048)], default=0), m._DECODE_M)")
    base = {k: v for k, v in os.environ.items() if k not in ("MXLLM_SKINNY_M", "MXLLM_NORM_FUSED_M")}
    out = subprocess.run([sys.executable, "-c", code], env={**base, **env}, capture_output=True, text=True, timeout=300,
                         cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert out.returncode == 0, out.stderr[-2000:]
    assert [int(v) for v in out.stdout.split()] == [rows, norm_rows, rows]


# (M, N, K): both sides of each line of the decode GEMMs' dispatch, as measured beside it in mxllm/ops/linear.py
DECODE_ROUTES = {
    "stream": [(1, 6144, 4096), (2, 128256, 4096), (8, 20480, 2048), (8, 8192, 6144), (9, 2048, 2048), (32, 12288, 2048),
               (16, 16384, 2048), (32, 20480, 2048), (16, 2048, 4096), (17, 16384, 4096), (9, 12288, 6144)],
    "half": [(1, 2048, 2048), (8, 2048, 8192), (1, 3584, 3072), (8, 512, 4096)],
    "skinny": [(1, 3072, 2048), (8, 3072, 2048), (2, 3584, 3072), (8, 2064, 8192), (1, 4096, 3072), (4, 512, 1536),
               (16, 64, 2048), (32, 1024, 2048), (32, 4096, 1536), (16, 3072, 3072), (12, 1024, 4096),
               (8, 16384, 2048), (8, 4096, 4096), (1, 128256, 4096), (4, 16384, 2048),
               (5, 128256, 2048), (3, 65536, 2560), (5, 128256, 1536), (7, 65536, 2048)],
    "": [(6, 128256, 2048), (4, 65536, 2560), (6, 128256, 1536), (17, 16384, 2048), (32, 14336, 2048), (17, 12288, 4096), (18, 28672, 4096), (9, 6144, 6144), (9, 28672, 8192),
         (17, 64, 2048), (32, 512, 1024), (16, 64, 4096), (13, 1024, 4096), (20, 2560, 2560), (9, 1024, 6144),
         (9, 4112, 1536), (33, 1024, 2048)],
}


@pytest.mark.parametrize("route,M,N,K", [(r, *s) for r, sizes in DECODE_ROUTES.items() for s in sizes])
def test_decode_routes(route, M, N, K):
    lin = sys.modules["mxllm.ops.linear"]
    assert lin._decode_route(M, N, K) == route


def test_what_the_skinny_entry_points_hand_on():
    """Behind the routes above: sizes that skinny_linear and w8_linear run on the GEMM that stays, both sides of each line."""
    from mxllm.ops import native

    on = [(3, 48, 2048), (8, 16384, 2048), (32, 3072, 2048), (9, 48, 4096), (16, 3072, 4096), (16, 4112, 4096)]
    off = [(2, 16384, 2048), (8, 3072, 4096), (9, 3088, 4096), (16, 4096, 4096), (17, 1024, 4096), (8, 3072, 3072), (12, 2048, 8192)]
    assert [s for s in on if not native().skinny_stays(*s)] == [] and [s for s in off if native().skinny_stays(*s)] == []
    assert all(native().w8_stays(*s) for s in ((3, 2048), (8, 4096), (5, 14336)))
    assert not any(native().w8_stays(*s) for s in ((2, 4096), (9, 2048), (4, 4608), (6, 14336)))


def test_swiglu_route_of_decode_rows():
    """With SwiGLU in the epilogue the GEMM that stays gains from fewer channels on, and past 16 rows at any."""
    wins = sys.modules["mxllm.ops.linear"]._stream_wins
    assert wins(8, 10240, 2048, True) and not wins(8, 8192, 2048, True) and not wins(8, 10240, 2048)
    assert wins(32, 16384, 2048, True) and not wins(32, 16384, 2048) and not wins(33, 16384, 2048, True)
    assert wins(12, 4096, 4096, True) and wins(16, 3584, 4096, True) and not wins(12, 4096, 4096)


def test_qkv_route_of_decode_rows():
    stream = sys.modules["mxllm.ops.linear"]._qkv_stream
    for M, K, norm, D, f8, want in ((1, 4096, False, 128, False, True), (8, 2048, False, 128, False, False),
                                    (9, 2048, False, 128, False, True), (1, 2048, True, 128, False, True),
                                    (1, 2048, False, 64, False, True), (8, 2048, False, 128, True, True),
                                    (16, 4096, False, 128, False, True), (17, 4096, False, 128, False, False),
                                    (5, 4096, True, 128, False, False)):
        assert stream(M, K, norm, D, f8) == want, (M, K, norm, D, f8)


def test_norm_route_of_decode_rows():
    wins = sys.modules["mxllm.ops.linear"]._norm_wins
    yes = [(1, 2048, 2048), (4, 3072, 2048), (1, 6144, 4096), (4, 4096, 4096), (3, 8192, 8192), (1, 10240, 8192)]
    no = [(1, 1024, 2048), (2, 4096, 4096), (1, 8192, 8192), (4, 4096, 14336), (1, 2048, 8192)]
    assert [s for s in yes if not wins(*s)] == [] and [s for s in no if wins(*s)] == []


def test_weight_gradient_rule():
    """Both sides of the lines that mxllm/ops/gemm.py draws for weight gradients outside the table (M, N, tokens)."""
    def on(M, N, T):
        return gemm._gains("tt", M, N, T)

    assert on(2048, 2048, 300) and on(2048, 2048, 3608) and on(2048, 2048, 5161) and on(3072, 2048, 5600)
    assert not on(2048, 2048, 4104) and not on(2048, 2048, 5600)
    assert on(128256, 2048, 768) and on(128256, 4096, 1280) and on(57344, 8192, 1544) and on(16384, 4096, 2304)
    assert not on(57344, 8192, 256) and not on(57344, 8192, 416) and not on(57344, 8192, 1536) and not on(8192, 28672, 2304) and not on(128256, 2048, 512)


def test_ragged_row_rules():
    """Both sides of the lines of ``gemm.rows_gain`` (rows, columns, K)."""
    def gain(M, N, K, form):
        return gemm.rows_gain(M, N, K, form != "nn", form == "swiglu")

    on = [(512, 8192, 28672, "tn"), (1100, 2048, 12288, "tn"), (1700, 128256, 8192, "tn"), (408, 28672, 8192, "nn"),
          (2635, 8192, 8192, "nn"), (1000, 8192, 57344, "nn"), (158, 128256, 8192, "tn"), (3328, 6144, 4096, "swiglu"), (1280, 16384, 2048, "swiglu"), (1377, 8192, 8192, "swiglu"),
          (3693, 10240, 8192, "swiglu"), (765, 21504, 4096, "swiglu")]
    off = [(559, 8192, 28672, "tn"), (768, 8192, 28672, "tn"), (2210, 128256, 8192, "tn"), (300, 28672, 8192, "nn"),
           (371, 28672, 8192, "nn"), (560, 8192, 57344, "nn"), (64, 128256, 8192, "tn"), (4013, 4096, 21504, "swiglu"), (1792, 10240, 4096, "swiglu"), (1105, 8192, 8192, "swiglu"),
           (3328, 10240, 8192, "swiglu"), (5120, 4096, 21504, "swiglu"), (512, 16384, 2048, "swiglu")]
    assert [s for s in on if not gain(*s)] == [] and [s for s in off if gain(*s)] == []


# (M, N, K): both sides of the lines of csrc/kernels/gemm_tile.hip mx_gemm_tile_plan
TILE_ON = [(9, 2048, 64), (33, 2048, 2048), (2709, 3072, 2048), (192 * 16, 192 * 16, 2048), (33, 2560, 4096), (32, 2048, 8192), (17, 4096, 14336), (430, 12288, 4096), (128, 8192, 8192), (256, 4096, 14336), (512, 2048, 12288),
           (40, 3360, 2048),
           (370, 3072, 2048), (290, 2048, 2048), (549, 2048, 8192), (150, 6144, 4096),
           # (too few tiles for most CUs, but .77 to .92 of the library's time)
           (1045, 2048, 2048), (1600, 2048, 2048), (2237, 2048, 2048), (667, 3072, 2048), (1079, 4096, 4096), (700, 6144, 4096), (540, 5120, 5120)]
TILE_OFF = [(192 * 16 + 1, 192 * 16, 2048), (255, 12288, 4096), (127, 8192, 8192), (257, 4096, 14336), (513, 2048, 12288), (40, 3368, 2048), (40, 2048, 2080),
            (32, 6144, 4096), (6, 128256, 2048), (2709, 16384, 2048), (2048, 128, 4096), (512, 256, 4096),
            # (the library was quicker by 4 to 18 %)
            (386, 6144, 4096), (430, 6144, 4096), (290, 4096, 4096), (370, 4096, 4096), (687, 4096, 4096), (290, 16384, 4096), (370, 16384, 4096),
            (370, 8192, 8192), (600, 8192, 8192), (370, 16384, 2048), (506, 5376, 4096), (10, 4096, 14336), (22, 6144, 16384), (48, 64, 4096), (300, 64, 4096)]


def test_tile_plan():
    from mxllm.ops import native

    assert [s for s in TILE_ON if gemm.tile_plan(*s) is None] == [] and [s for s in TILE_OFF if gemm.tile_plan(*s) is not None] == []
    assert gemm.tile_plan(48, 28672, 4096, True) and not gemm.tile_plan(48, 28672, 4096) and not gemm.tile_plan(48, 57344, 8192, True)
    assert not gemm.tile_plan(130, 28672, 4096, True) and gemm.tile_plan(200, 28672, 4096, True) and gemm.tile_plan(135, 21504, 4096, True) and not gemm.tile_plan(16, 7168, 16384, True)
    assert gemm.tile_plan(9, 1024, 4096, True)[1] <= 8  # (in 16 parts the sum and its activation are what lasts)
    assert native().gemm_tile_plan(0, 64, 64, False) == native().gemm_tile_plan(1 << 40, 64, 64, False) == -1


@pytest.mark.parametrize("N,K", [(64, 4096), (128, 4096), (256, 4096), (64, 2048), (128, 2048), (256, 8192)])
def test_gates_are_not_cut_along_k(N, K):
    """A gate's or a router's sums are one sum in order at any number of rows: short prompts and long ones round alike."""
    for M in (9, 17, 32, 33, 48, 300, 511, 512, 700, 2048, 4096):
        for swiglu in (False, True):
            plan = gemm.tile_plan(M, N, K, swiglu)
            assert plan is None or plan[1] == 1, (M, swiglu, plan)
    assert gemm.tile_plan(48, N + 256, 8192)[1] > 1  # (past them they are)


def test_tile_plan_is_one_turn():
    """Whatever the sizes: tiles and parts of K that the CUs hold at once, four 64s of K a part and more."""
    import random

    tiles = [(64, 64, 256), (64, 128, 256), (128, 128, 256), (128, 192, 256), (128, 256, 256), (160, 192, 256), (192, 192, 256)]
    r, seen = random.Random(0), set()
    for _ in range(4000):
        M, N, K = int(2 ** r.uniform(0, 13)), 16 * int(2 ** r.uniform(0, 11)), 64 * int(2 ** r.uniform(0, 9))
        plan = gemm.tile_plan(M, N, K)
        if plan:
            tm, tn, most = tiles[plan[0]]
            assert -(-M // tm) * -(-N // tn) * plan[1] <= most and (plan[1] == 1 or K // 64 >= 4 * plan[1]), (M, N, K, plan)
            seen.add(plan[0])
    assert seen == set(range(7))
