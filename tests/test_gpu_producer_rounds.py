"""Reverse kernels of the sLSTM whose producer wave runs its first round of three steps in front of its loop: sequence
lengths around one, two and three rounds, with the outputs stored by the compute waves and by the producer wave."""
import pytest

from parity import check_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stores", ["0", "1"])
@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 6, 7, 11])
@pytest.mark.parametrize("dtype,D", [("bfloat16", 64), ("float16", 96)])
def test_slstm_reverse_at_the_edges_of_the_rounds(gpu, monkeypatch, dtype, D, T, stores):
    monkeypatch.setenv("FRNN_PRODUCER_STORES", stores)
    print(f"case producer rounds slstm {dtype} B5 T{T} N2 D{D} stores={stores}", flush=True)
    check_case(gpu, "slstm", 5, T, 2, D, dtype, "hip_fused", seed=T)
