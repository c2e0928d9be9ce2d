// The head dim 256 build of paged_prefill.hip (paged in every pool format, or packed): see the note at the top
// of that file.
#define LITEKV_HD 256
#include "paged_prefill.hip"
