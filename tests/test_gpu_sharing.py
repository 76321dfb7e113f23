"""What several graphs, calls and host threads share: the device copies of a model's weights, the plain product's kept
workspace, the pinned ring that inputs and results travel through; kernels between which a graph's size decides."""
import ctypes as C
import os
import tempfile
import threading

import numpy as np
import pytest

from aspen_amd import api, models as M
from tests import helpers as H

pytestmark = pytest.mark.gpu


def in_threads(jobs):
    """Runs the jobs side by side and raises what one of them raised."""
    failed = []

    def guarded(job):
        try:
            job()
        except BaseException as e:                 # noqa: B902  (handed on below)
            failed.append(e)
    threads = [threading.Thread(target=guarded, args=(job,)) for job in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    assert not any(t.is_alive() for t in threads)
    if failed:
        raise failed[0]


class Product:
    """Operands of one plain product on the device, and what comes out of it."""

    def __init__(self, m, n, k, seed, offset=0):
        L = api.lib()
        rng = np.random.default_rng(seed)
        self.shape, self.ldc = (m, n, k), -(-m // 4) * 4
        self.A, self.B = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
        self.d = [L.aspen_hip_alloc(x) for x in (self.A.nbytes + 16, self.B.nbytes, n * self.ldc * 4)]
        assert all(self.d)
        self.a = self.d[0] + 4 * offset
        assert L.aspen_hip_h2d(self.a, self.A.ctypes.data, self.A.nbytes) == 0
        assert L.aspen_hip_h2d(self.d[1], self.B.ctypes.data, self.B.nbytes) == 0
        a, b = self.A.astype(np.float64), self.B.astype(np.float64)
        self.exact = b @ a.T
        # one rounding per 16 K positions in each of the two running sums, a few behind them, 2^-24 of the magnitudes each
        self.bound = (2 * (k // 16) + 8) * 2.0 ** -24 * (np.abs(b) @ np.abs(a).T)

    def run(self):
        (m, n, k), L = self.shape, api.lib()
        out = np.zeros((n, self.ldc), dtype=np.float32)
        assert L.aspen_hip_sgemm(m, n, k, self.a, k, self.d[1], k, self.d[2], self.ldc, None, 0) == 0, L.aspen_hip_last_error()
        assert L.aspen_hip_d2h(out.ctypes.data, self.d[2], out.nbytes) == 0
        return out[:, :m]

    def check(self):
        out = self.run()
        assert np.all(np.abs(out - self.exact) <= self.bound), self.shape

    def close(self):
        for d in self.d:
            api.lib().aspen_hip_free(d)


def test_products_one_after_the_other_in_the_kept_workspace(gpu):
    """Larger, smaller and larger again than what the workspace holds, nothing given back in between; the smaller ones find the
    remains of others behind their own rows, and everything still fits after the workspace was released."""
    shapes = [(200, 90, 64), (700, 300, 320), (33, 31, 96), (700, 300, 320), (1500, 64, 512), (129, 127, 1056)]
    products = [Product(*s, seed=i) for i, s in enumerate(shapes)]
    try:
        api.lib().aspen_hip_release_workspaces()
        for p in products + products[::-1]:
            p.check()
        api.lib().aspen_hip_release_workspaces()
        api.lib().aspen_hip_release_workspaces()
        products[1].check()
    finally:
        for p in products:
            p.close()


def test_products_of_two_host_threads(gpu):
    """Two threads call the product at the same time: one has the kept workspace, the other one takes its own.  Every result
    against its own 64-bit sums."""
    products = [Product(600, 500, 512, 1), Product(64, 1500, 768, 2), Product(900, 40, 1024, 3)]
    try:
        in_threads([lambda p=p: [p.check() for _ in range(20)] for p in products] + [lambda: [api.lib().aspen_hip_release_workspaces() for _ in range(20)]])
    finally:
        for p in products:
            p.close()


@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_first_operand_of_any_float_alignment(gpu, offset):
    """A begins 4, 8 or 12 bytes behind a 16-byte boundary (a view of a larger matrix)."""
    p = Product(70, 45, 160, 9, offset)
    try:
        p.check()
    finally:
        p.close()


def test_matrices_of_two_host_threads_travel_whole(gpu):
    """Two threads send and fetch matrices of several rings' length at the same time, a third one small ones: bit for bit."""
    L = api.lib()
    for f in (L.aspen_hip_dense_host_to_device, L.aspen_hip_dense_host_to_device_ordered):
        f.argtypes = [C.c_void_p, C.c_uint32, C.c_void_p, C.c_uint32, C.c_size_t]
    L.aspen_hip_dense_device_to_host.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, C.c_uint32, C.c_size_t]

    def job(rows, ld, columns, times, seed):
        d = L.aspen_hip_alloc(ld * columns * 4)
        assert d
        try:
            for i in range(times):
                x = np.random.default_rng(seed + i).integers(0, 2 ** 32, rows * columns, dtype=np.uint32)
                back, up = np.zeros_like(x), L.aspen_hip_dense_host_to_device if i & 1 else L.aspen_hip_dense_host_to_device_ordered
                assert up(d, ld, x.ctypes.data, rows, columns) == 0
                assert L.aspen_hip_dense_device_to_host(back.ctypes.data, d, ld, rows, columns) == 0
                assert np.array_equal(back, x), (rows, columns, i)
        finally:
            L.aspen_hip_free(d)
    in_threads([lambda: job(85, 96, 70001, 4, 10), lambda: job(64, 64, 100003, 4, 20), lambda: job(3, 4, 777, 60, 30)])


@pytest.mark.parametrize("mode", [api.MODE_LAYERS, api.MODE_DATAFLOW], ids=["layers", "dataflow"])
def test_two_graphs_of_one_model_hold_a_layer_in_either_form(gpu, monkeypatch, mode):
    """A fully connected layer in 128 x 32 tiles (a batch of 9: weights as floats) and in 64 x 64 ones (a batch of 80: as three
    terms) of the same model, in turns, and again with other weights."""
    from oracle import cpu
    monkeypatch.setenv("ASPEN_GPU_WEIGHT_STREAM_BYTES", "0")
    monkeypatch.setenv("ASPEN_GPU_NARROW_TILES", "0")
    cfg = "[net]\nheight=4\nwidth=4\nchannels=64\n\n[connected]\noutput=200\nactivation=relu\n\n[connected]\noutput=24\nactivation=linear\n\n"
    layers = M.parse_cfg(cfg)
    tens = M.synth_weights(layers, 81, "he")
    big = H.GpuNet(cfg, tens, 80, 0, min_ninst=4, mode=mode)
    nasm, pool, dse = api.Nasm(big.dnn, 9, 0, 4), api.RPool(), api.DseGroup(1, mode)
    dse.set_rpool(pool)
    try:
        assert [big.nasm.info(1)["variant"], nasm.info(1)["variant"]] == [2, 4]
        for turn in range(2):
            x = (M.synth_input(layers, 82 + turn, 80, 0, "token_ids") * 2.0 - 1.0).astype(np.float32)
            want, want9 = cpu.run_network(layers, tens, x, 80, 0), cpu.run_network(layers, tens, x[:9].copy(), 9, 0)
            for _ in range(2):
                big.run(x)
                pool.add_nasm_raw_input(nasm, x[:9].copy())
                dse.run()
                dse.wait(nasm)
                dse.stop()
                for l in (1, 2):
                    assert H.rel_l2(big.layer(l), want[l]) <= H.REL_L2_TOL and H.rel_l2(nasm.layer_output(l), want9[l]) <= H.REL_L2_TOL, (turn, l)
            if turn == 0:
                tens = M.synth_weights(layers, 83, "he")
                path = tempfile.mktemp(suffix=".bin")
                M.write_aspen_data(path, tens)
                api.lib().apu_load_dnn_data_from_file(big.dnn.h, path.encode())
                os.unlink(path)
    finally:
        dse.destroy()
        pool.destroy()
        nasm.destroy()
        big.close()


@pytest.mark.parametrize("batch", [1, 4, 5, 9])
def test_ordered_transformer_graphs_agree_with_launches_per_layer(gpu, batch):
    """Two blocks of BERT-base, 128 tokens each, from graphs of little parallelism on.  The sums are formed in one order everywhere, so
    the persistent kernel agrees with one launch per layer to a rounding or two per layer: ten layers deep, 2^-24 each, 2^-20 in all."""
    cfg = M.bert_cfg(2, 768, 12, 3072)
    layers = M.parse_cfg(cfg)
    tens = M.synth_weights(layers, 91, "gpt")
    x = M.synth_input(layers, 91, batch, 128, "embeddings")
    api.lib().aspen_keep_layer_outputs(0)
    try:
        net = H.GpuNet(cfg, tens, batch, 128, min_ninst=192, mode=api.MODE_LAYERS)
        dse = api.DseGroup(1, api.MODE_DATAFLOW)
        dse.set_rpool(net.rpool)
        try:
            net.run(x)
            last = net.nasm.num_ldata - 1
            want = net.layer(last).copy()
            for _ in range(3):
                net.rpool.reset_nasm(net.nasm)
                dse.run()
                dse.wait(net.nasm)
                dse.stop()
                assert H.rel_l2(net.layer(last), want) <= 2.0 ** -20
            assert net.rpool.run_stats() == {"executed": net.nasm.num_ninst, "double_runs": 0, "aborted": 0}
        finally:
            dse.destroy()
            net.close()
    finally:
        api.lib().aspen_keep_layer_outputs(1)
