"""LDS that lanes of one wave trade without a barrier of the work-group: the hardware keeps a wave's accesses in order, the
compiler only where the source says so.  It says so with a wave barrier, which the assembly shows.  No device is needed."""
import re

from test_host_registers import compiled


def body_of(source, name):
    text = compiled(source)[1]
    for kernel in sorted(set(re.findall(r"^(_Z\w*%s\w*):" % name, text, re.M))):
        body = text[text.index("\n" + kernel + ":"):]
        yield kernel, body[:body.index(".Lfunc_end")]


def test_scales_of_a_new_int8_row_are_in_place_before_others_read_them():
    # stored 16 bits a lane, read 32 bits a lane by others: two types, so nothing but the barrier orders them
    seen = 0
    for kernel, body in body_of("decode_attn_mfma.hip", "decode_attn_mfma_i8h_kernel"):
        pending = False
        for event in re.findall(r"^\s+(ds_write_b16|ds_read\w*|s_barrier)\b|^\s+; (wave barrier)", body, re.M):
            event = event[0] or event[1]
            seen += event == "ds_write_b16"
            assert not (pending and event.startswith("ds_read")), kernel
            pending = event == "ds_write_b16" or pending and not event.endswith("barrier")
    assert seen >= 4, "two step kernels, each in a long walk and in ranges of one page a wave"


def test_rows_of_q_and_of_the_output_are_traded_in_order():
    # f16 chunks with one tile a wave: q comes and the outputs leave row by row, 16 bytes a lane
    kernels = list(body_of("prefill_attn.hip", "prefill_attn_kernelILi0ELi1E"))
    assert len(kernels) == 2, "cut and not"
    for kernel, body in kernels:
        last, trades, traded_q = None, 0, False
        for access, barrier in re.findall(r"^\s+(ds_write_b128|ds_read_b128|s_barrier)\b|^\s+; (wave barrier)", body, re.M):
            now = access.split("_")[1] if access.startswith("ds_") else None
            traded_q |= access == "s_barrier"
            assert not (last == "write" and now == "read"), kernel
            # (behind q other images are read beside the rows of V that are cleared)
            assert traded_q or not (last == "read" and now == "write"), kernel
            trades += last == "write" and bool(barrier)
            last = now
        assert trades == 3, "eight rows of q, the other eight, the output"
