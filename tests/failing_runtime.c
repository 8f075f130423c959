// Stands in for the HIP runtime's calls of mesh_ctx_create (loaded before the
// library, which then binds to these): one device, a stream and pinned memory, whose
// device address cannot be had.  Counts what is created and what is given back.
#include <stddef.h>
#include <stdlib.h>

enum
{
	OK = 0,
	INVALID = 1
};

int live_streams, live_pinned;

int hipGetDeviceCount(int *n) { return *n = 1, OK; }
int hipSetDevice(int d) { return d == 0 ? OK : INVALID; }
int hipGetLastError(void) { return OK; }
int hipStreamCreateWithFlags(void **s, unsigned flags)
{
	(void)flags;
	*s = malloc(1);
	++live_streams;
	return OK;
}
int hipStreamDestroy(void *s)
{
	free(s);
	--live_streams;
	return OK;
}
int hipHostMalloc(void **p, size_t n, unsigned flags)
{
	(void)flags;
	*p = malloc(n);
	++live_pinned;
	return OK;
}
int hipHostFree(void *p)
{
	free(p);
	--live_pinned;
	return OK;
}
int hipHostGetDevicePointer(void **d, void *p, unsigned flags)
{
	(void)d, (void)p, (void)flags;
	return INVALID;
}
