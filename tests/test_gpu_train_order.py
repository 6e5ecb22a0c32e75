"""Order of the rows in classifier training (GPU): every epoch takes every row once. With a learning rate
of 0 each epoch's loss is the mean over all rows, whatever their order and batches; a row
taken twice for another moves it by some 1/rows of its value."""
import numpy as np
import pytest

from rabbitqcplus_amd import learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,batch", [(1, 1), (1000, 100), (4096, 64), (500_000, 50_000)])
def test_every_epoch_takes_every_row_once(rows, batch):
    print(f"[rows {rows} batch {batch}]", flush=True)
    rng = np.random.default_rng(95)
    X = (4.0 * rng.standard_normal((rows, 16))).astype(np.float32)
    y = rng.integers(0, 2, rows).astype(np.float32)
    mlp = learned.Mlp(0)
    mlp.set_params(learned.init_params(5))
    mlp.reset_optimizer()
    mlp.set_data(X, y)
    losses = np.asarray(mlp.train(6, batch=batch, lr=0.0, seed=3), np.float64)
    z = np.asarray(mlp.forward(X), np.float64)
    mean = np.mean(np.maximum(z, 0.0) - z * y + np.log1p(np.exp(-np.abs(z))))
    # float sums of a batch's 256-row parts and of at most 64 batches: some 100 roundings of 6e-8
    assert np.all(np.abs(losses - mean) <= 1e-5 * mean), losses / mean - 1.0
