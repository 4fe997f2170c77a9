// Host entries of the block-tridiagonal offsets (spitfire_amd/csrc/gf_btd_index.h) for tests/test_btd_index.py.
#include "../../spitfire_amd/csrc/gf_btd_index.h"

extern "C" {
long btd_values_host(int nb, int bs) { return gfa::btd_values(nb, bs); }
long btd_sup_host(int nb, int bs, int i) { return gfa::btd_sup(nb, bs, i); }
}
