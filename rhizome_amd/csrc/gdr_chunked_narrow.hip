// gdr_chunked_narrow.hip -- the chunked prefill kernel's instances with 16
// state rows per workgroup, compiled in a unit of their own: the kernel
// source is gdr_chunked.hip, whose launch code calls chunked_go_narrow and
// chunked_narrow_counter defined here.
#define RHZ_CHUNKED_NARROW_TU 1
#include "gdr_chunked.hip"
