#include "simt.h"
