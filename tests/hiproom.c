/* hipMalloc with a limit on one allocation's size, in front of the runtime's own. */
#include <stddef.h>
long room = -1; /* largest allocation allowed; negative: any */
int (*real)(void **, size_t);
int hipMalloc(void **p, size_t n) { return room >= 0 && (long)n > room ? 2 : real(p, n); }
