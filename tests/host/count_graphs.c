/* Counts graph instantiations: loaded with RTLD_GLOBAL before the library, its
 * hipGraphInstantiate is the one that the library binds to. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

static int count;

int graphs_instantiated(void) { return count; }

int hipGraphInstantiate(void** exec, void* graph, void* node, char* log, size_t size)
{
    typedef int (*fn)(void**, void*, void*, char*, size_t);
    fn next = (fn)dlsym(RTLD_NEXT, "hipGraphInstantiate");
    count++;
    return next ? next(exec, graph, node, log, size) : 1;
}
