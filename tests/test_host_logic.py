"""Host logic of the C ABI without a GPU: api.hip compiled for the host against stand-ins for the HIP runtime and the kernel
launchers (host_runtime.cpp).  What is allocated, given back, kept and refused; nothing is computed."""
import ctypes as C
import os
import subprocess

import pytest

from tests.conftest import ROOT, load_pkg

L = load_pkg("_lib")
OOM = 2      # OMEGA_ERR_OOM


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "host_logic.so")
    csrc = os.path.join(ROOT, "omega-ai_amd", "csrc")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-w", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                           "-D__align__(n)=__attribute__((aligned(n)))", "-DHIP_SYMBOL(x)=((const void *)(x))",
                           "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"), "-I" + csrc, "-o", so,
                           "-x", "c++", os.path.join(csrc, "api.hip"), os.path.join(ROOT, "tests", "host_runtime.cpp")])
    lib = C.CDLL(so)
    for name, (res, args) in L.SIGNATURES.items():
        if hasattr(lib, name):
            getattr(lib, name).restype, getattr(lib, name).argtypes = res, args
    lib.host_live_bytes.restype = C.c_size_t
    lib.host_take_log.restype = C.c_char_p
    return lib


class Layer:
    """A layer over the stand-ins; the buffers of its caller are addresses that nothing follows."""

    def __init__(self, lib, dtype="f32", d=256, H=256, E=4, K=2, Es=1, T_max=0):
        self.lib, self.ctx, self.h = lib, C.c_void_p(), C.c_void_p()
        assert lib.omega_hip_ctx_create(0, C.byref(self.ctx)) == 0
        cfg = L.MoEConfigStruct(T_max, d, E, K, H, Es, 1, 1, L.DTYPE_BF16 if dtype == "bf16" else L.DTYPE_F32, L.ROUTER_EXACT)
        assert lib.omega_moe_create(self.ctx, C.byref(cfg), C.byref(self.h)) == 0
        self.x, self.g, self.out = 0x1000, 0x2000, 0x3000

    def forward(self, T):
        return self.lib.omega_moe_forward(self.h, self.x, T, self.out)

    def back(self, T):
        return self.lib.omega_moe_backward(self.h, self.x, self.g, T, self.out)

    def stages(self, T):
        """The stages up to the up product, one by one."""
        return [self.lib.omega_moe_router(self.h, self.x, T), self.lib.omega_moe_dispatch(self.h, self.x, T),
                self.lib.omega_moe_experts_up(self.h, self.x, T)]

    def grad_status(self):
        import numpy as np
        return self.lib.omega_moe_get_grad(self.h, L.W_GATE_BIAS, 0, np.empty(64, np.float32).ctypes.data, 0)

    def log(self):
        return self.lib.host_take_log().decode().splitlines()

    def close(self):
        assert self.lib.omega_moe_destroy(self.h) == 0 and self.lib.omega_hip_ctx_destroy(self.ctx) == 0


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_a_backward_workspace_is_there_whole_or_not_at_all(lib, dtype):
    """Whichever allocation of the backward pass runs out of memory, everything that it took before is given back, nothing that
    follows works on a part of it, and the next call finds no error left behind."""
    for n in range(1, 100):
        m = Layer(lib, dtype)
        assert m.forward(8) == 0
        before = lib.host_live_count(), lib.host_live_bytes()
        lib.host_fail_allocation(n)
        st = m.back(8)
        lib.host_fail_allocation(0)
        if st == 0:
            break
        assert st == OOM and (lib.host_live_count(), lib.host_live_bytes()) == before, n
        assert m.lib.omega_moe_set_training(m.h, 1) == 0
        m.log()
        assert m.stages(8) == [0, 0, 0], n          # no error of the failed allocation, and ...
        assert not any("keep=1" in s or "without" in s for s in m.log()), n    # ... nothing kept where there is no room
        assert m.forward(8) == 0 and m.back(8) == 0 and "without" not in "".join(m.log()) and m.grad_status() == 0
        m.close()
    assert n > 10      # (every allocation had its turn)
    m.close()
    assert lib.host_live_count() == 0


def test_an_fp32_training_forward_without_room_keeps_nothing(lib):
    """... and the gradients of an earlier backward pass, which are not part of the workspace."""
    for n in range(1, 100):
        m = Layer(lib)
        assert m.forward(8) == 0
        before = lib.host_live_count(), lib.host_live_bytes()
        assert lib.omega_moe_set_training(m.h, 1) == 0
        lib.host_fail_allocation(n)
        assert m.forward(8) == 0, n
        lib.host_fail_allocation(0)
        if any("keep=1" in s for s in m.log()):
            break
        assert (lib.host_live_count(), lib.host_live_bytes()) == before, n
        assert m.grad_status() != 0          # no backward pass has run
        assert m.forward(8) == 0 and m.back(8) == 0 and "backward_f32 kept=1" in m.log()
        lib.host_fail_allocation(20)         # (a forward pass of more tokens: its own workspace, then the backward pass's)
        assert m.forward(64) == 0 and m.grad_status() == 0
        lib.host_fail_allocation(0)
        assert "product_f32 op=0 gather=1 keep=0" in m.log()
        m.close()
    assert n > 8
    m.close()


def test_a_failed_forward_leaves_no_batch_to_go_back_through(lib):
    """A training forward that found no room for the backward workspace routed nothing: the index buffers are an earlier
    batch's, and a backward pass that formed its addresses from them would read past their end.  It is refused."""
    m = Layer(lib, "bf16", T_max=32)
    assert m.forward(8) == 0 and lib.omega_moe_set_training(m.h, 1) == 0
    lib.host_fail_allocation(3)
    assert m.forward(16) == OOM
    lib.host_fail_allocation(0)
    assert m.back(16) == 1 and m.back(8) == 1
    assert m.forward(16) == 0 and m.back(16) == 0
    m.close()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_backward_rows_can_be_read_behind_a_backward_pass_only(lib, dtype):
    """dh (bf16 layers) and dlogits of a workspace that a training forward allocated, and of one that has grown since the last
    backward pass, hold nothing yet."""
    import numpy as np
    m = Layer(lib, dtype)
    host = np.empty(1 << 18, np.float32)

    def read():
        return {w: lib.omega_moe_get_workspace(m.h, w, 8, host.ctypes.data) for w in ((3, 4) if dtype == "bf16" else (4,))}

    assert lib.omega_moe_set_training(m.h, 1) == 0 and m.forward(8) == 0
    assert set(read().values()) == {1}
    assert m.back(8) == 0
    assert set(read().values()) == {0}
    assert m.forward(8) == 0 and set(read().values()) == {0}     # the last backward pass's, until the next
    assert m.forward(64) == 0
    assert set(read().values()) == {1}
    ms = C.c_float()
    assert lib.omega_moe_time_backward(m.h, m.x, m.g, 64, m.out, 0, 1, C.byref(ms)) == 0 and set(read().values()) == {0}
    m.close()


@pytest.mark.parametrize("T,tile", [(1, 32), (1023, 32), (1024, 128), (3000, 128)])
def test_fp32_rows_are_padded_to_the_tile_in_use(lib, T, tile):
    """xg, a and y hold every expert's rows in whole tiles of the height that a batch of T tokens takes; batches of fewer
    tokens, which may take the lower one, need no more."""
    d, H, E, K, Es = 64, 32, 48, 3, 2
    m = Layer(lib, d=d, H=H, E=E, K=K, Es=Es)
    before = lib.host_live_bytes()
    assert m.forward(T) == 0
    per_row = (2 * d + H) * 4 + 4       # xg, y, a and the row's token
    rest = T * (5 * K * 4 + d * 4 + 4) + (T // 16 + 17) * E * 4 + (T * K // 32 + E + Es * (T // 32 + 1)) * 16
    rows = (T * K // tile + E + Es * -(-T // tile)) * tile
    assert rows * per_row <= lib.host_live_bytes() - before <= rows * per_row + rest
    assert rows >= max((t * K // h + E + Es * -(-t // h)) * h for t in (T, 1000, 1) if t <= T for h in ([32, 128] if t >= 1024 else [32]))
    m.close()


@pytest.mark.parametrize("dtype,training", [("f32", 1), ("f32", 0), ("bf16", 1), ("bf16", 0)])
def test_time_backward_times_the_pass_of_its_mode(lib, dtype, training):
    """After a training forward every timed pass finds h1, h3 and the probabilities kept, also in an fp32 layer, whose pass
    uses them up; computing them again between the passes is not timed (the stand-in's clock counts launches: one a pass)."""
    m = Layer(lib, dtype)
    assert lib.omega_moe_set_training(m.h, training) == 0 and m.forward(8) == 0
    m.log()
    ms = C.c_float()
    for warmup, iters in ((2, 3), (0, 1)):
        assert lib.omega_moe_time_backward(m.h, m.x, m.g, 8, m.out, warmup, iters, C.byref(ms)) == 0
        passes = [s for s in m.log() if s.startswith("backward_")]
        assert passes == [f"backward_{dtype} kept={training}"] * (warmup + iters) and ms.value == 1.0
        assert m.forward(8) == 0 and m.log()
    m.close()


@pytest.mark.parametrize("dtype,d,E", [("bf16", 256, 4), ("bf16", 4096, 8), ("bf16", 2048, 16), ("bf16", 768, 7), ("f32", 68, 5),
                                       ("f32", 33, 3)])
def test_expert_blocks_of_the_optimiser_start_on_a_cache_line(lib, dtype, d, E):
    """Gradients, moments and master weights of the experts start on 128 bytes, the blocks they are part of on 16, whatever the
    widths of the gate; the layer gives all of them back."""
    m = Layer(lib, dtype, d=d, E=E)
    assert m.forward(8) == 0 and m.back(8) == 0
    for step in (1, 2):
        assert lib.omega_moe_acc_grad(m.h, 1.0) == 0
        m.log()
        assert lib.omega_moe_update_adamw(m.h, 1e-3, 0.9, 0.999, 0.0, step) == 0
        assert m.log()[-1] == "adamw block 0 experts 0"
        assert m.forward(8) == 0 and m.back(8) == 0
    m.close()
    assert lib.host_live_count() == 0


def test_reads_into_device_memory_go_through_the_kernel(lib):
    """The library does not load without it: there is no other way that a build which lost it could fall back to."""
    import numpy as np
    m = Layer(lib, "bf16")
    assert m.forward(8) == 0 and m.back(8) == 0
    p = C.c_void_p()
    assert lib.omega_hip_malloc(m.ctx, 256 * 256 * 4, C.byref(p)) == 0
    for get, which, line in ((lib.omega_moe_get_weights, L.W_W1, "param_read of a packed image"), (lib.omega_moe_get_weights, L.W_GATE, "param_read"),
                             (lib.omega_moe_get_grad, L.W_W1, "param_read")):
        m.log()
        assert get(m.h, which, 0, p, 1) == 0 and m.log() == [line]
        host = np.empty(256 * 256, np.float32)
        assert get(m.h, which, 0, host.ctypes.data, 0) == 0 and line not in m.log()
    assert lib.omega_hip_free(m.ctx, p) == 0
    m.close()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_the_kernel_stores_to_memory_of_its_own_device_only(lib, dtype):
    """Where the caller's buffer is host memory, another device's, unknown or too short, the runtime copies - or refuses - as it
    always did, and leaves no error behind."""
    import numpy as np
    m = Layer(lib, dtype)
    n = 256 * 256 * 4
    assert m.forward(8) == 0 and m.back(8) == 0
    p = C.c_void_p()
    assert lib.omega_hip_malloc(m.ctx, n, C.byref(p)) == 0
    lib.host_move_to_device.argtypes = [C.c_void_p, C.c_int]
    reads = [(lib.omega_moe_get_weights, L.W_W1, n // (2 if dtype == "bf16" else 1)), (lib.omega_moe_get_weights, L.W_GATE_BIAS, 16), (lib.omega_moe_get_grad, L.W_W2, n)]
    host = np.empty(n, np.uint8)

    def read(get, which, dst):
        m.log()
        st = get(m.h, which, 0, dst, 1)
        return st, [s for s in m.log() if s != "unpack"]

    for get, which, size in reads:
        st, log = read(get, which, p.value + n - size)              # to the last byte
        assert st == 0 and len(log) == 1 and log[0].startswith("param_read")
        assert read(get, which, host.ctypes.data) == (0, ["copy"])
        assert read(get, which, p.value + n - size + 4) == (3, [])  # past the end: OMEGA_ERR_HIP
        lib.host_move_to_device(p, 1)
        assert read(get, which, p.value) == (0, ["copy"])
        lib.host_move_to_device(p, 0)
        assert m.forward(8) == 0
    live = lib.host_live_count()
    read(lib.omega_moe_get_weights, L.W_W1, host.ctypes.data)
    assert lib.host_live_count() == live
    assert lib.omega_hip_free(m.ctx, p) == 0
    m.close()


def test_queues_that_could_not_be_made_are_made_by_the_next_pass(lib):
    """A forward pass of a few tokens leaves the tile kernels' queues to the backward pass; where their launch fails they are still
    those of an earlier batch, and no product may run on them."""
    m = Layer(lib, "bf16")
    ms = C.c_float()
    for back in (m.back, lambda T: lib.omega_moe_time_backward(m.h, m.x, m.g, T, m.out, 0, 1, C.byref(ms))):
        assert m.forward(64) == 0 and m.back(64) == 0 and m.forward(8) == 0
        m.log()
        lib.host_fail_launch(b"index")
        assert back(8) == 3 and not any(s.startswith("backward") for s in m.log())      # OMEGA_ERR_HIP
        assert back(8) == 0
        log = m.log()
        assert log.index("index") < log.index("backward_bf16 kept=0")
        assert back(8) == 0 and "index" not in m.log()
    m.close()


@pytest.mark.parametrize("dtype,T,training", [("f32", 8, 0), ("bf16", 8, 0), ("bf16", 64, 0), ("bf16", 65, 0), ("bf16", 8, 1)])
def test_a_timed_forward_pass_is_one(lib, dtype, T, training):
    """Stage 5 of time_stage makes the launches of omega_moe_forward, and leaves what it leaves."""
    m = Layer(lib, dtype)
    assert lib.omega_moe_set_training(m.h, training) == 0
    for _ in range(2):
        m.log()
        assert m.forward(T) == 0
        want = m.log()
    ms = C.c_float()
    assert lib.omega_moe_time_stage(m.h, 5, m.x, T, m.out, 1, 2, C.byref(ms)) == 0
    assert m.log() == 3 * want and ms.value == len(want)
    assert m.back(T) == 0
    m.close()


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 12, 15, 16, 31, 33, 54, 60, 64, 127])
@pytest.mark.parametrize("mats", [1, 2, 5, 8, 17, 24])
def test_tiles_of_weight_gradients_are_dealt_evenly(lib, n, mats):
    """Every tile of every matrix to one workgroup, the XCDs' totals next to alike, and each one's share a run in rising order; of a
    matrix of 32 tiles or more an eighth, rounded up or down."""
    seen, totals = set(), []
    per = -(-n * mats // 8) + (1 if n < 32 else 0)      # the launch's workgroups per XCD
    for x in range(8):
        got = [lib.host_wgrad_tile(n, mats, x, j) for j in range(per + 3)]
        assert set(got[per:]) == {-1}
        got = [t for t in got if t >= 0]
        assert got == sorted(got) and not seen & set(got)
        seen |= set(got)
        totals.append(len(got))
        if n >= 32:
            for m in range(mats):
                run = [t for t in got if t // n == m]
                assert len(run) in (n // 8, -(-n // 8)) and run == list(range(run[0], run[0] + len(run)))
    assert seen == set(range(n * mats)) and max(totals) - min(totals) <= (1 if n >= 32 else 2)


@pytest.mark.parametrize("dtype,up", [("bf16", "experts_bf16 which=0 keep=0"), ("f32", "product_f32 op=0 gather=1 keep=0")])
def test_the_index_is_launched_unless_the_up_product_makes_it(lib, dtype, up):
    """A forward pass of a few tokens leaves the dispatch index to its up product; whoever else asks for the index gets its launch, and a pass whose up
    product was not launched leaves no index."""
    m = Layer(lib, dtype)
    assert m.forward(8) == 0 and "index" not in m.log()
    assert m.back(8) == 0 and m.log().count("index") == (1 if dtype == "bf16" else 0)     # (the work queues of the backward pass)
    assert m.stages(8) == [0, 0, 0] and m.log().count("index") == 1
    assert m.forward(600) == 0 and m.log().count("index") == 1
    lib.host_fail_launch(up.encode())
    assert m.forward(8) != 0 and m.lib.omega_moe_experts_up(m.h, m.x, 8) != 0 and m.lib.omega_moe_experts_down(m.h, 8) != 0
    assert m.forward(8) == 0
    m.close()
