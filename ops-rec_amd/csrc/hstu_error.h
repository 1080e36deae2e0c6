// The calling thread's last error text, shared by the host translation units of the library.
#pragma once

namespace hstu {

// formats the text that hstu_last_error() returns on this thread and hands `code` back
int set_error(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
// compute units of the current device, looked up once per device; HSTU_OK, or the code of set_error without a usable device
int compute_units(int* out);

}  // namespace hstu
