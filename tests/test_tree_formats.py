"""Exported trees in both formats (lists per tree; packed node arrays) give the
same predictions, also from trees that are one leaf."""

import json

import numpy as np
import pytest

from tilec import tune


@pytest.mark.parametrize("depth", [1, 4])
def test_formats_agree(tmp_path, depth):
    from sklearn.ensemble import GradientBoostingRegressor
    rng = np.random.default_rng(1)
    X = rng.normal(size=(300, 5))
    y = np.where(X[:, 0] > 3, X[:, 1], X[:, 2] ** 2)
    m = GradientBoostingRegressor(n_estimators=30, max_depth=depth, min_samples_leaf=1, random_state=0).fit(X, y)
    tune.export(m, str(tmp_path / "m.json"))
    packed = json.loads((tmp_path / "m.json").read_text())
    lists = {k: packed[k] for k in ("learning_rate", "init", "n_features")}
    lists["trees"] = [{"left": t.children_left.tolist(), "right": t.children_right.tolist(),
                       "feature": t.feature.tolist(), "threshold": t.threshold.tolist(),
                       "value": t.value[:, 0, 0].tolist()} for t in (e.tree_ for e in m.estimators_[:, 0])]
    leaf = {"left": [-1], "right": [-1], "feature": [-2], "threshold": [-2.0], "value": [0.25]}
    Xt = rng.normal(size=(70, 5))
    want = m.predict(Xt)
    np.testing.assert_allclose(tune.TreeModel(packed).predict(Xt), want, rtol=1e-12, atol=1e-12)
    np.testing.assert_allclose(tune.TreeModel(lists).predict(Xt), want, rtol=1e-12, atol=1e-12)
    lists["trees"].append(leaf)
    np.testing.assert_allclose(tune.TreeModel(lists).predict(Xt), want + 0.25 * lists["learning_rate"], rtol=1e-12,
                               atol=1e-12)
