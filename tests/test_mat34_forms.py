"""mat34 takes every form of twelve numbers that float() takes one by one."""
import decimal

import numpy as np
import pytest
import torch

from multiviewdynrecon_amd.render import mat34

BASE = [0.5 * k - 2 for k in range(12)]
FORMS = {
    "list": BASE, "tuple": tuple(BASE), "float32": np.array(BASE, np.float32), "float16": np.array(BASE, np.float16),
    "strided": np.repeat(BASE, 2)[::2], "longer": np.array(BASE + [7.0]), "column": np.array(BASE)[:, None],
    "decimals": np.array([decimal.Decimal(k) for k in BASE], object), "text": np.array([str(k) for k in BASE]),
    "complex": np.array(BASE, complex), "tensor": torch.tensor(BASE), "bfloat16": torch.tensor(BASE).bfloat16(),
}


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("form", FORMS)
def test_forms(form):
    m = mat34(FORMS[form])
    assert list(m.rot) + list(m.trans) == BASE


@pytest.mark.parametrize("m", [np.zeros((3, 4)), np.zeros(11), [0.0] * 11])
def test_refused(m):
    with pytest.raises((TypeError, ValueError)):
        mat34(m)
