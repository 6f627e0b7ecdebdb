"""Minimal stand-in for the reference's ``my_utils`` package: only the ``Logger`` the operator
calls (``my_utils/my_log/log_performance.py:7-56``).  Messages go to ``log/application.log``
unless ``ANCHOR_ATTN_LOG=0`` is exported."""
import datetime
import locale
import os
import time


class Logger:
    log_file_path = "log/application.log"
    enabled = os.environ.get("ANCHOR_ATTN_LOG", "1") != "0"

    @classmethod
    def set_log_file_path(cls, path: str = None):
        cls.log_file_path = os.path.join("log", path or str(time.time()))

    @classmethod
    def log(cls, message):
        """``message``: a string, or a function that returns it - called with the file open, so that a message which has to be
        fetched from the GPU is waited for last."""
        if not cls.enabled:
            return
        try:
            file = cls._opened()
            try:
                if callable(message):
                    message = message()
                stamp = datetime.datetime.now().isoformat(" ", "milliseconds")
                line = f"{stamp} - {message}\n".encode(locale.getpreferredencoding(False))
                while line:
                    line = line[os.write(file, line):]
            finally:
                os.close(file)
        except OSError as e:
            print(f"Unable to write to log file: {e}")

    # The operator logs on every call, and on a few thousand tokens the next call's launch waits for that: a line is one write to a descriptor, 4 us
    # of the host (a text file object and a look for the folder each time: 12).  Calls in a row, 2048 tokens with 14/2 heads of 64: 29.1 us -> 28.1.
    @classmethod
    def _opened(cls):
        flags = os.O_WRONLY | os.O_CREAT | os.O_APPEND | os.O_CLOEXEC
        try:
            return os.open(cls.log_file_path, flags, 0o666)
        except FileNotFoundError:
            os.makedirs(os.path.dirname(cls.log_file_path), exist_ok=True)
            return os.open(cls.log_file_path, flags, 0o666)

    log.__func__.takes_function = True  # (a function in this one's place may know strings only)

    @classmethod
    def log_error(cls, m: str):
        cls.log(f"ERROR: {m}")

    @classmethod
    def log_warning(cls, m: str):
        cls.log(f"WARNING: {m}")

    @classmethod
    def log_info(cls, m: str):
        cls.log(f"INFO: {m}")
