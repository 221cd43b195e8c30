import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
	sys.path.insert(0, ROOT)


def pytest_configure(config):
	config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu where there is one)")


def pytest_collection_modifyitems(config, items):
	try:
		import torch

		has_gpu = torch.cuda.is_available()
	except Exception:
		has_gpu = False
	if has_gpu:
		return
	skip = pytest.mark.skip(reason="no GPU in this environment")
	for item in items:
		if "gpu" in item.keywords:
			item.add_marker(skip)
