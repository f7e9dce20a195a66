"""GPU radiance cache (rt_cache_* through the C ABI) against the oracle's
FP64 model of the same network (oracle/mlp.c, itself pinned by finite
differences): forward outputs, loss and gradients of the BF16/MFMA kernels,
then online training on a known function.

Bar: with the oracle emulating the GPU's BF16 storage points, gradients
agree to a relative L2 error below 2e-2 (FP32 accumulation order and BF16
re-rounding of intermediate values remain); outputs to 1e-2 relative."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def records(n, seed):
    rng = np.random.default_rng(seed)
    r = np.zeros((n, 12), np.float32)
    r[:, :3] = rng.uniform(0.02, 0.98, (n, 3))
    nr = rng.normal(size=(n, 3))
    r[:, 3:6] = nr / np.linalg.norm(nr, axis=1, keepdims=True)
    vd = rng.normal(size=(n, 3))
    r[:, 6:9] = vd / np.linalg.norm(vd, axis=1, keepdims=True)
    r[:, 9] = rng.uniform(0, 1, n)
    return r


def rel_err(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@pytest.fixture(scope="module")
def small(rt, gpu_ctx, orc):
    kw = dict(levels=4, log2_table=10, base_res=4, per_level_scale=2.0, batch=1024, seed=3)
    cache = rt.RadianceCache(gpu_ctx, (0, 0, 0), (1, 1, 1), **kw)
    cfg = orc.cache_cfg(4, 10, 4, 2.0, (0, 0, 0), (1, 1, 1))
    # larger grid features than the default init so the encoding matters
    mlp, grid = cache.get_params()
    rng = np.random.default_rng(11)
    grid = rng.uniform(-0.5, 0.5, grid.shape).astype(np.float32)
    cache.set_params(mlp, grid)
    yield cache, cfg, mlp, grid
    cache.close()


def test_level_table_matches_oracle(small):
    cache, cfg, _, _ = small
    inf = cache.info()
    assert [inf.res[l] for l in range(4)] == [cfg.res[l] for l in range(4)]
    assert [inf.dense[l] for l in range(4)] == [cfg.dense[l] for l in range(4)]


def test_forward_matches_oracle(small, orc):
    cache, cfg, mlp, grid = small
    rec = records(1000, 1)
    y_gpu = cache.query(torch.from_numpy(rec).cuda())
    torch.cuda.synchronize()
    y_gpu = y_gpu.cpu().numpy()
    _, _, _, y = orc.cache_loss_grad(cfg, mlp, grid, rec, np.zeros((1000, 3), np.float32), emulate_bf16=True,
                                     want_grad=False)
    y_ref = np.maximum(y, 0)
    err = np.abs(y_gpu - y_ref)
    assert np.max(err) <= 1e-2 * max(1.0, np.max(np.abs(y_ref)))
    assert rel_err(y_gpu, y_ref) < 1e-2


def test_gradients_match_oracle(small, orc):
    cache, cfg, mlp, grid = small
    rec = records(1000, 2)
    rng = np.random.default_rng(4)
    tgt = rng.uniform(0, 2, (1000, 3)).astype(np.float32)
    loss, mg, gg = cache.gradients(torch.from_numpy(rec).cuda(), torch.from_numpy(tgt).cuda())
    l_ref, mg_ref, gg_ref, _ = orc.cache_loss_grad(cfg, mlp, grid, rec, tgt, emulate_bf16=True)
    print(f"[cache grads] loss gpu {loss:.6f} oracle {l_ref:.6f}; mlp rel err {rel_err(mg, mg_ref):.2e}; "
          f"grid rel err {rel_err(gg, gg_ref):.2e}", flush=True)
    assert abs(loss - l_ref) <= 1e-2 * l_ref
    assert rel_err(mg, mg_ref) < 2e-2
    assert rel_err(gg, gg_ref) < 2e-2
    # per layer, so a wrong operand layout in one GEMM cannot hide
    for l in range(5):
        off, size = l * 4096, (1024 if l == 4 else 4096)
        assert rel_err(mg[off:off + size], mg_ref[off:off + size]) < 3e-2, l
    # unused output columns get no gradient
    assert np.all(mg[16384:].reshape(64, 16)[:, 3:] == 0)


def test_online_training_fits_a_smooth_field(rt, gpu_ctx):
    """Adam (lr 1e-2) on a smooth radiance field of position and normal:
    the relative L2 loss falls by more than an order of magnitude."""
    cache = rt.RadianceCache(gpu_ctx, (0, 0, 0), (1, 1, 1), levels=16, log2_table=19, batch=65536, seed=1)

    def field(r):
        p, n = r[:, :3], r[:, 3:6]
        base = 0.6 + 0.4 * np.sin(6 * p[:, 0]) * np.cos(5 * p[:, 1]) + 0.3 * p[:, 2]
        return np.stack([base * (0.7 + 0.3 * n[:, 2]), base * 0.8, base * (0.6 + 0.2 * n[:, 0])], 1).astype(np.float32)

    losses = []
    for step in range(300):
        rec = records(65536, 100 + step)
        tgt = field(rec)
        losses.append(cache.train_step(torch.from_numpy(rec).cuda(), torch.from_numpy(tgt).cuda()))
    print(f"[cache train] loss {losses[0]:.4f} -> {losses[-1]:.5f}", flush=True)
    assert np.isfinite(losses).all()
    assert losses[-1] < losses[0] / 10
    # held-out error
    rec = records(20000, 9999)
    y = cache.query(torch.from_numpy(rec).cuda()).cpu().numpy()
    t = field(rec)
    assert np.sqrt(np.mean((y - t) ** 2)) < 0.1
    cache.close()


def last_cells(levels, log2_table, base, scale):
    """Grid features that are zero but for the last entries of every level: the
    last table entries of a hashed one, the last row of cells of a dense one."""
    g = np.zeros((levels, 1 << log2_table, 2), np.float32)
    for l in range(levels):
        res = int(np.floor(base * float(np.float32(scale)) ** l))
        dense = (res + 1) ** 3 <= 1 << log2_table
        end = (res + 1) ** 3 if dense else 1 << log2_table
        k = res + 1 if dense else 2
        g[l, end - k:end] = np.random.default_rng(12 + l).uniform(2, 4, (k, 2))
    return g.reshape(-1)


@pytest.mark.parametrize("levels,log2_table,base,scale", [(1, 8, 2, 1.0), (3, 9, 7, 1.7), (5, 12, 4, 2.0), (16, 10, 16, 1.38)])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 1000, 70001])
@pytest.mark.parametrize("last", [False, True])
def test_query_sizes_and_level_counts(rt, gpu_ctx, orc, levels, log2_table, base, scale, n, last):
    """Strips of 16 rows with remainders, level counts that end inside a
    feature tile, dense levels that fill their table (res 7 and 512 entries),
    positions on the box's faces (the last cell's clamped corners); with
    `last`, only the last entries of a level are not zero and most rows lie at
    the far corner, so that a wrong half of a pair load there is the answer.

    The oracle rounds at the same places, so answers agree to float rounding
    but for a row in which a sum rounds to the other BF16 neighbour (2^-8 of
    one of 64 activations; 8.5e-4 of 0.19 measured at most).  Such rows are rare:
    an RMS of 2e-5 of 0.067 at most.  The last entry of each level zeroed moves the
    answers by an RMS of 8e-4 to 3e-3, with `last` by 2e-3 to 0.1."""
    cache = rt.RadianceCache(gpu_ctx, (0, 0, 0), (1, 1, 1), levels=levels, log2_table=log2_table, base_res=base,
                             per_level_scale=scale, batch=256, seed=3)
    cfg = orc.cache_cfg(levels, log2_table, base, scale, (0, 0, 0), (1, 1, 1))
    mlp, grid = cache.get_params()
    grid = (last_cells(levels, log2_table, base, scale) if last
            else np.random.default_rng(11).uniform(-0.5, 0.5, grid.shape).astype(np.float32))
    cache.set_params(mlp, grid)
    rec = records(n, 1)
    if last:
        rec[:, :3] = np.where(np.random.default_rng(3).random((n, 3)) < 0.5, 1.0, 1.0 - 0.1 * rec[:, :3])
    rec[:: 7, 0] = 1.0
    rec[3:: 7, 1] = 0.0
    rec[5:: 7, 2] = 1.0
    y = cache.query(torch.from_numpy(rec).cuda()).cpu().numpy()
    m = min(n, 2000)
    at = np.r_[:m // 2, n - (m - m // 2):n]
    ref = orc.cache_loss_grad(cfg, mlp, grid, rec[at], np.zeros((m, 3), np.float32), emulate_bf16=True,
                              want_grad=False)[3]
    ref = np.maximum(ref, 0)
    err = np.abs(y[at] - ref)
    assert np.max(err) <= 1e-2 * np.max(ref)
    assert np.sqrt(np.mean(err ** 2)) <= 1e-3 * np.sqrt(np.mean(ref ** 2))
    cache.close()


@pytest.mark.parametrize("levels,log2_table,base,scale", [(1, 8, 2, 1.0), (3, 9, 7, 1.7), (5, 12, 4, 2.0), (16, 15, 16, 1.38)])
@pytest.mark.parametrize("n", [1, 15, 17, 64, 65, 257, 1000])
def test_gradient_sizes_and_level_counts(rt, gpu_ctx, orc, levels, log2_table, base, scale, n):
    """Strips of 16 rows, chunks of 64 and runs of 256 with remainders, level
    counts that end inside a feature tile, nearly as many distinct cells in a run
    as its merge table holds (16 levels), positions on the box's faces (both
    corners of a pair in one cell).  Five BF16 storage points in series, each
    off by at most one rounding (2^-8) from the oracle's: 5 * 2^-8 < 2e-2."""
    cache = rt.RadianceCache(gpu_ctx, (0, 0, 0), (1, 1, 1), levels=levels, log2_table=log2_table, base_res=base,
                             per_level_scale=scale, batch=1000, seed=3)
    cfg = orc.cache_cfg(levels, log2_table, base, scale, (0, 0, 0), (1, 1, 1))
    mlp, grid = cache.get_params()
    grid = np.random.default_rng(11).uniform(-0.5, 0.5, grid.shape).astype(np.float32)
    cache.set_params(mlp, grid)
    rec = records(n, 5)
    rec[:: 7, 0] = 1.0
    rec[3:: 7, 1] = 0.0
    rec[5:: 7, 2] = 1.0
    tgt = np.random.default_rng(6).uniform(0, 2, (n, 3)).astype(np.float32)
    loss, mg, gg = cache.gradients(torch.from_numpy(rec).cuda(), torch.from_numpy(tgt).cuda())
    l_ref, mg_ref, gg_ref, _ = orc.cache_loss_grad(cfg, mlp, grid, rec, tgt, emulate_bf16=True)
    assert abs(loss - l_ref) <= 1e-2 * l_ref
    assert rel_err(mg, mg_ref) < 2e-2
    assert rel_err(gg, gg_ref) < 2e-2
    cache.close()
